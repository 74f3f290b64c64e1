// Guarded bf16 GEMM for gfx950: C[M,N] = A[M,K] * B[K,N], row-major, fp32
// accumulation in ascending k, bf16 (round-to-nearest-even) output.
//
// MFMA-bound: 2*M*N*K flop. One work-group of 512 threads (8 wavefronts) owns one
// 256x256 tile of C and walks K in steps of 64 through two LDS buffers:
//   global -> LDS       buffer_load ... lds: every wave-wide load moves 64 x 16 bytes straight
//                       into 1 KiB of LDS, no registers and no LDS store instructions in
//                       between. Lane l of a load fills the l-th 16-byte slot of that KiB and
//                       is free in what it fetches, so the tiles are kept unpadded and
//                       XOR-swizzled: the slot a piece lands in is its natural slot XOR a few
//                       bits of its row, chosen so that every fragment read below touches
//                       each LDS bank once.
//                       A tile: [256 rows][64 k], two rows to a 256-byte line of sixteen
//                       slots, slot = (row & 1) * 8 + ((k / 8) ^ (line & 7)).
//                       B tile: as it sits in memory, [64 k][256 cols], sixteen 32-byte granules
//                       to a row, granule = (col / 16) ^ ((k & 3) * 2 + ((k >> 3) & 1)).
//   LDS -> MFMA         v_mfma_f32_16x16x32_bf16; wave (wm, wn) of the 2x4 wave grid
//                       accumulates a 128x64 sub-tile = 8x4 blocks of 16x16
// An MFMA operand wants eight consecutive k per lane. A has them contiguous in memory; for B
// (k is the strided dimension) the transposing LDS read of gfx950, ds_read_b64_tr_b16, turns
// four rows of sixteen columns into four k of one column per lane, two of them per fragment.
// Every element of C is summed in an order that M, N, K and the number of compute units decide: from k = 0 on,
// or, where K is divided (SplitK), part by part, the parts' sums added in their order, whether they are
// computed by several work-groups or, without memory for that, by one: a replayed tile is bit-identical, and so is the product of
// the same data at another address, under capture or with little memory left.
//
// Under this load the device runs against its power limit (all operands zero, when next to nothing
// switches, 8192^3 takes 567 us, normally distributed ones 782 on the same box and code), so
// energy is time:
//   - blocks of 16x16 rather than 32x32: MFMAs alone, operands in registers, reach 2.0 PFLOP/s on
//     normally distributed operands with the one and 1.78 with the other (2.4 both on zeroes; an MFMA
//     of 32x32 reads and writes twice the accumulators per flop). The sums are bit for bit the same.
//   - neighbouring MFMAs share an operand (the columns of every other row of blocks run backwards): 1 %.
//   - the loads of a step are spread evenly over half of it: next to every fourth MFMA 727 us, next to
//     every second 733, every one 750.
// 8192^3 782 -> 725 us per launch, 4096^3 102.0 -> 94.8 (1.52 and 1.45 PFLOP/s).
//
// Guard: the tile is computed in registers and written once at the end, so a
// work-group may give up at any K step without side effects. The preempt word is
// checked at entry and then every kPollSteps K steps: wave 0 requests it with a vector load
// at the top of the step and looks at it in front of the barrier the loop has anyway, so
// nobody waits for it; a flushed tile leaves its progress byte untagged and is redone by
// the replay. The tile is written out through LDS (64-bit stores of four rows of a column,
// transposing reads back), whole rows of 128 bytes per eight lanes.
// Work-group ids are remapped so that the 32 CUs of one XCD (ids equal modulo 8 land on one
// XCD) work on neighbouring tiles and share A/B panels in that XCD's L2.
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <utility>

#include "hip_hal.h"
#include "xsched/hip/hal.h"

using namespace xsched::preempt;

namespace xsched::hip
{

namespace gemm
{

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 LdsS16x4;
typedef __attribute__((address_space(3))) void LdsVoid;
typedef __attribute__((address_space(3))) volatile uint32_t LdsVolatileWord;
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int kLargeTile = 256;     // edge of the large tile of C (M and N)
constexpr int kThreeQuarterRows = 192, kHalfRows = 128;   // rows of the large tile where fewer than 256 of them divide M better
constexpr int kSmallTile = 128;     // edge of the small one
constexpr int kTinyTile = 64;       // and of the smallest
constexpr int kStepK = 64;          // K per step
constexpr int kPollSteps = 4;       // K steps between two looks at the preempt word
constexpr int kXcds = 8;
constexpr int kGroupRows = 4;       // tile rows walked together
constexpr int kMaxK = 1 << 22;      // 32-bit byte offsets inside a 256-row panel of A

/// Two floats rounded to nearest-even bf16 (NaNs quieted), `lo` in the low half: the
/// conversion instruction of gfx950 (v_cvt_pk_bf16_f32), which gives bit for bit what the
/// integer formula (u + 0x7FFF + ((u >> 16) & 1)) >> 16, NaN -> (u >> 16) | 0x40 gives (a GPU
/// test compares the two over products that hit ties, overflow, denormals, infinities and
/// NaNs).
__device__ __forceinline__ uint32_t f32x2_to_bf16x2_rne(float lo, float hi)
{
    const bf16x2 pair = __builtin_convertvector(f32x2 { lo, hi }, bf16x2);
    return __builtin_bit_cast(uint32_t, pair);
}

// Work-group id -> number of its work. Ids with equal (id % 8) run on one XCD; each XCD gets a
// contiguous run of the n numbers.
__device__ __forceinline__ uint32_t WorkOf(uint32_t wg, uint32_t n)
{
    const uint32_t xcd = wg % kXcds, whole = n / kXcds, more = n % kXcds;   // `more` XCDs get one more
    return xcd * whole + min(xcd, more) + wg / kXcds;
}

// Tile number t -> tile coordinates, in bands of kGroupRows tile rows.
__device__ __forceinline__ void TileAt(uint32_t t, uint32_t tiles_m, uint32_t tiles_n,
                                       uint32_t &tm, uint32_t &tn)
{
    const uint32_t band = kGroupRows * tiles_n;
    const uint32_t band_id = t / band;
    const uint32_t first_row = band_id * kGroupRows;
    const uint32_t rows = min((uint32_t)kGroupRows, tiles_m - first_row);
    const uint32_t in_band = t - band_id * band;
    tm = first_row + in_band % rows;
    tn = in_band / rows;
}

#define XS_PIN __builtin_amdgcn_sched_barrier(0)
#define XS_WAIT_GLOBAL_LOADS __builtin_amdgcn_s_waitcnt(0x0F70) /* vmcnt(0), nothing else */

// What the matrices have to be like is kFit:
//   kExact      M, N multiples of the tile, K of kStepK, matrices aligned to 16 bytes
//   kEdges      rows of A and B that start on 16-byte boundaries (their lengths in memory, lda and ldb,
//               are multiples of 8; M, N, K and C are any): a 16-byte piece begins inside the matrix
//               or lies outside. Pieces outside are fetched from somewhere
//               inside (their row or column of C is not stored); behind K the fragments are
//               masked to zero, which adds nothing to a sum
//   kUnaligned  any N >= 8, any alignment to the element: pieces start at any multiple of two
//               bytes, which the loads into LDS do not take: they come through registers
//               (a tile or two in flight) and are stored to the same places. Only
//               the last K step can reach behind the end of a matrix: a piece that does is fetched
//               from the matrix's last 16 bytes instead and shifted into place.
enum class Fit { kExact, kEdges, kUnaligned };

typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef s16x8 s16x8_any __attribute__((aligned(2)));

/// The 16 bytes of v moved down by d (0..15) bytes, zeroes behind them.
__device__ __forceinline__ u32x4 ShiftDownBytes(u32x4 v, uint32_t d)
{
    const u32x4 zero = { 0, 0, 0, 0 };
    v = d & 8 ? __builtin_shufflevector(v, zero, 2, 3, 4, 4) : v;
    v = d & 4 ? __builtin_shufflevector(v, zero, 1, 2, 3, 4) : v;
    return u32x4 { __builtin_amdgcn_alignbyte(v.y, v.x, d & 3), __builtin_amdgcn_alignbyte(v.z, v.y, d & 3),
                   __builtin_amdgcn_alignbyte(v.w, v.z, d & 3), __builtin_amdgcn_alignbyte(0u, v.w, d & 3) };
}

/// Whether rows of C start on 16-byte boundaries (uniform).
__device__ __forceinline__ bool WholeRowPieces(const uint16_t *C, int N) { return (((uintptr_t)C | (uint32_t)N * 2u) & 15) == 0; }

/// Eight columns of a row of C, as far as they are inside. `whole`: WholeRowPieces().
template <Fit kFit>
__device__ __forceinline__ void StoreEight(uint16_t *C, size_t row, size_t col, int M, int N, bool whole, s16x8 eight)
{
    uint16_t *const at = C + row * (size_t)N + col;
    if constexpr (kFit == Fit::kExact) {
        __builtin_nontemporal_store(eight, (s16x8 *)at);
    } else if (row < (size_t)M) {
        if (kFit == Fit::kEdges && whole) {
            if (col < (size_t)N) __builtin_nontemporal_store(eight, (s16x8 *)at);
        } else if (col + 8 <= (size_t)N) {
            *(s16x8_any *)at = eight;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) if (col + e < (size_t)N) at[e] = (uint16_t)eight[e];
        }
    }
}

/// What a K step of the large-tile kernel requests: nothing, a tile that is not the last one, or the
/// last one.
enum TileRequest { kNoTile, kAnyButLast, kTheLast };

// Two LDS buffers and ONE barrier per K step. A step is two k slices of 32. While the MFMAs of the
// first one run, the fragments of the second are read from buffer t % 2, and tile t + 1 lands in the
// other buffer (its loads were issued over the slice before); after the barrier buffer t % 2 is free:
// next to the MFMAs of the second slice the first fragments of tile t + 1 are read and the loads of
// tile t + 2 go out.
//
// kTileM x kTileN is the tile of C, kWavesM x kWavesN the wave grid over it; a wave owns
// kBlocksM x kBlocksN blocks of 16x16. Built for 256 x 256 with 2x4 waves (8x4 blocks
// per wave), for exact shapes and for ragged ones (kEdges): there the last tile's loads, the last
// step and the stores look at the edges, and the steps before are the same code (4000^3 146 us on
// 128 x 128 tiles, 106 on these). For 192 x 256 and 128 x 256, with the same waves of 6x4 and 4x4 blocks: a step
// takes 1.08 and 0.82 us of a full round where 256 rows take 1.36, so a round that 256 rows leave half empty is shorter by up to
// a quarter (who takes which: QuickestPlan()). More bytes go through LDS per flop (11 % and 33 %), which is why they are not taken
// where whole rounds of 256 rows fit. And for 128 x 128 with 2x2 waves (4x4 blocks), exact shapes only: 64 KiB
// of LDS and 4 waves, so two work-groups share a compute unit and one computes while the other
// waits for its first loads or writes out. That is what outputs of 257 to 512 such tiles want,
// which are two rounds for the four-stage kernel below (its 130 KiB let a unit have one group), and
// what short K wants, where a tile is little more than its first loads and its write-out
// (per command: 368 tiles at K = 192 10.1 -> 7.3 us, at 2048 33.5 -> 28.9; 276 at 4096 55.1 -> 50.1;
// 1023 at 128 16.5 -> 10.7).
// Four waves of 128x128 on the large tile (a third fewer LDS reads, one wave per SIMD, accumulators
// in AGPRs) take 732 us for 8192^3 where eight take 725, and 595 against 567 on zeroes: nothing runs
// beside their barrier.
//
// (The body is a device function: the host pass cannot parse the buffer-resource builtins
// and would silently drop the launch stub of a kernel that uses them directly.)
template <bool kGuard, Fit kFit, int kTileM, int kTileN, int kWavesM, int kWavesN>
__device__ __forceinline__
void GemmBf16Body(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                  uint16_t *__restrict__ C, int M, int N, int K, int lda, int ldb, const XGuardArgs &g)
{
    static_assert(kFit != Fit::kUnaligned, "loads go straight into LDS");
    constexpr int kWaves = kWavesM * kWavesN;
    constexpr int kBlocksM = kTileM / (16 * kWavesM);
    constexpr int kBlocksN = kTileN / (16 * kWavesN);
    constexpr int kMfmas = kBlocksM * kBlocksN;          // per wave and 32-wide k slice
    constexpr int kReads = kBlocksM + kBlocksN;          // fragments of a slice
    constexpr int kABytes = kTileM * kStepK * 2;          // one A tile in LDS
    constexpr int kBBytes = kStepK * kTileN * 2;          // one B tile
    constexpr int kALoads = kABytes / 1024 / kWaves;     // wave-wide 1 KiB loads per wave and tile
    constexpr int kBLoads = kBBytes / 1024 / kWaves;
    constexpr int kLoads = kALoads + kBLoads;
    constexpr int kLoadEvery = kMfmas / kLoads;          // one load next to so many MFMAs
    constexpr int kBRowBytes = kTileN * 2;                // one k row of the B tile
    constexpr int kBSlotsPerRow = kBRowBytes / 16;
    constexpr int kBRowsPerLoad = 64 / kBSlotsPerRow;
    static_assert(kBlocksN == 4, "the block index is XORed into the granule number as two bits");
    static_assert(kBRowBytes >= 256, "a granule number has the three bits that are XORed");
    static_assert(kLoadEvery * kLoads <= kMfmas && 2 * kReads <= kMfmas, "loads and reads pair up with the MFMAs of a slice");
    // One LDS object for everything, the word the waves agree on a poll through included:
    // with a second object the compiler attaches alias scopes to the LDS accesses and then
    // makes every fragment read wait for all global loads that are on their way into LDS.
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * (kABytes + kBBytes) + 16];
    uint32_t &guard_word = *(uint32_t *)(lds + 2 * (kABytes + kBBytes));
    uint8_t *const As0 = lds;
    uint8_t *const Bs0 = lds + 2 * kABytes;

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave / kWavesN;
    const uint32_t wn = wave % kWavesN;

    uint32_t tm, tn;
    const uint32_t tiles_m = ((uint32_t)M + kTileM - 1) / kTileM, tiles_n = ((uint32_t)N + kTileN - 1) / kTileN;
    TileAt(WorkOf(blockIdx.x, tiles_m * tiles_n), tiles_m, tiles_n, tm, tn);
    const size_t m0 = (size_t)tm * kTileM, n0 = (size_t)tn * kTileN;
    const int steps = kFit == Fit::kExact ? K / kStepK : (K + kStepK - 1) / kStepK;
    const int rest = K - (steps - 1) * kStepK;           // K values of the last step

    // ---- global -> LDS: lane l of wave-wide load q fills LDS slot 64 q + l (16 bytes) ----
    // Byte offsets of what each lane fetches, relative to the first element of the tile.
    uint32_t a_off[kALoads], b_off[kBLoads];
    auto a_k = [&](int i) -> uint32_t { return ((lane & 7) ^ ((4 * (wave * kALoads + i) + (lane >> 4)) & 7)) * 8; };   // first k of its piece
    auto b_k = [&](int i) -> uint32_t { return kBRowsPerLoad * (wave * kBLoads + i) + lane / kBSlotsPerRow; };
#pragma unroll
    for (int i = 0; i < kALoads; ++i) {
        uint32_t row = 2 * (4 * (wave * kALoads + i) + (lane >> 4)) + ((lane >> 3) & 1);
        if (kFit != Fit::kExact && m0 + row >= (size_t)M) row = (uint32_t)((size_t)M - 1 - m0);   // not stored
        a_off[i] = (row * (uint32_t)lda + a_k(i)) * 2;
    }
#pragma unroll
    for (int i = 0; i < kBLoads; ++i) {
        const uint32_t k = b_k(i), slot = lane % kBSlotsPerRow;
        uint32_t col = ((slot >> 1) ^ ((k & 3) << 1 | ((k >> 3) & 1))) * 16 + (slot & 1) * 8;
        if (kFit != Fit::kExact && n0 + col >= (size_t)N) col = 0;                                // not stored
        b_off[i] = (k * (uint32_t)ldb + col) * 2;
    }
    const uint16_t *const a_tile = A + m0 * (size_t)lda;   // + 64 columns per step
    const uint16_t *const b_tile = B + n0;               // + 64 rows per step

    // Byte offset of load number idx (A first, then B) within its matrix's part of a K step. In the
    // last step pieces behind K come from k = 0 of the step instead.
    auto piece_off = [&](int idx, bool last) -> uint32_t {
        if (idx < kALoads) {
            if (kFit == Fit::kExact || !last) return a_off[idx];
            const uint32_t k = a_k(idx);
            return k < (uint32_t)rest ? a_off[idx] : a_off[idx] - k * 2;
        }
        if (kFit == Fit::kExact || !last) return b_off[idx - kALoads];
        const uint32_t k = b_k(idx - kALoads);
        return k < (uint32_t)rest ? b_off[idx - kALoads] : b_off[idx - kALoads] - k * (uint32_t)ldb * 2;
    };
    // Load number idx of the tile of K step `step` into buffer `buf`.
    auto load_piece = [&](int buf, int step, int idx, bool last) {
        if (idx < kALoads) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(a_tile + (size_t)step * kStepK), 0, 0x7fffffff, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)(As0 + buf * kABytes + (wave * kALoads + idx) * 1024), 16, piece_off(idx, last), 0, 0, 0);
        } else {
            const int i = idx - kALoads;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(b_tile + (size_t)step * kStepK * ldb), 0, 0x7fffffff, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)(Bs0 + buf * kBBytes + (wave * kBLoads + i) * 1024), 16, piece_off(idx, last), 0, 0, 0);
        }
    };
    auto load_tile = [&](int buf, int step) {
        if (kFit != Fit::kExact && step == steps - 1) {
#pragma unroll
            for (int idx = 0; idx < kLoads; ++idx) load_piece(buf, step, idx, true);
        } else {
#pragma unroll
            for (int idx = 0; idx < kLoads; ++idx) load_piece(buf, step, idx, false);
        }
    };

    // ---- LDS -> fragments ----
    // A: lane reads row a_row0 + 16 i, piece 4 ks + (lane >> 4). 16 rows further is 8 lines
    // further: the same swizzle bits, so one base address serves all blocks of the wave.
    const uint32_t a_row0 = 16 * kBlocksM * wm + (lane & 15);
    const uint32_t a_line = a_row0 >> 1;
    const uint32_t a_base = a_line * 256 + ((((lane & 1) << 3) | ((lane >> 4) ^ (a_line & 7))) << 4);
    auto read_a = [&](int buf, int ks, int i) {
        return *(const bf16x8 *)(As0 + buf * kABytes + (a_base ^ (ks << 6)) + i * 2048);
    };
    // B sits in LDS as it sits in memory, [k][n]. The transposing read hands lane l of every 16
    // lanes the element (l & 3) of what lanes 4 * j + (l >> 2), j = 0..3, of the same 16 point
    // at: with lane r pointing at row (r >> 2), columns 4 * (r & 3) .. + 3, lane l receives
    // column l of rows 0..3. Two reads give the eight consecutive k of one fragment. The rows
    // a lane points at all have the same swizzle bits (k & 3 and bit 3 of k are fixed per lane).
    const uint32_t b_row = 8 * (lane >> 4) + ((lane & 15) >> 2);
    const uint32_t b_swz = ((lane & 15) >> 2) << 1 | ((lane >> 4) & 1);
    const uint32_t b_base = b_row * kBRowBytes + (((kBlocksN * wn) ^ b_swz) << 5) + 4 * (lane & 3) * 2;
    auto read_b = [&](int buf, int ks, int j) {
        const uint8_t *p = Bs0 + buf * kBBytes + ks * 32 * kBRowBytes + (b_base ^ (j << 5));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)p);
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)(p + 4 * kBRowBytes));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    bf16x8 fa[2][kBlocksM], fb[2][kBlocksN];
    // Fragment number n of slice ks into set ks, in the order in which the MFMAs want them.
    auto read_frag = [&](int buf, int ks, int n) {
        if (n < kBlocksN) fb[ks][n] = read_b(buf, ks, n);
        else fa[ks][n - kBlocksN] = read_a(buf, ks, n - kBlocksN);
    };

    f32x4 acc[kBlocksM][kBlocksN];
#pragma unroll
    for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j) acc[i][j] = f32x4 { 0.f, 0.f, 0.f, 0.f };
    auto mfma = [&](int ks, int n) {
        const int i = n / kBlocksN, j = i & 1 ? kBlocksN - 1 - n % kBlocksN : n % kBlocksN;
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[ks][i], fb[ks][j], acc[i][j], 0, 0, 0);
    };

    // A lane's fragment of slice ks holds k = 32 ks + 8 (lane / 16) + 0..7 of the step, for A and
    // for B alike: everything from `rest` on becomes zero.
    auto mask_behind_k = [&](int ks) {
        const int valid = rest - (32 * ks + 8 * (int)(lane >> 4));
        u32x4 m;
#pragma unroll
        for (int d = 0; d < 4; ++d) m[d] = valid >= 2 * d + 2 ? 0xFFFFFFFFu : valid == 2 * d + 1 ? 0xFFFFu : 0u;
#pragma unroll
        for (int i = 0; i < kBlocksM; ++i) fa[ks][i] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fa[ks][i]) & m);
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j) fb[ks][j] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fb[ks][j]) & m);
    };

    // (the guard's words are requested first: waiting for them waits for nothing else)
    const XGuardBlock guard(g, blockIdx.x, &guard_word);
    const XGuardEntry entry = kGuard ? guard.EnterBegin() : XGuardEntry {};
    XS_PIN;
    load_tile(0, 0);

    if (kGuard) {
        if (!guard.EnterEnd(entry)) {
            XS_WAIT_GLOBAL_LOADS; // nothing may still be on its way into LDS when the group is gone
            return;
        }
    }

    XS_WAIT_GLOBAL_LOADS;
    __syncthreads();
    load_tile(1, steps > 1 ? 1 : 0);
#pragma unroll
    for (int n = 0; n < kReads; ++n) read_frag(0, 0, n);

    // One K step. The polling form (every kPollSteps-th step of a guarded launch) is a body of
    // its own: its branches split the step into several scheduling regions and put the address
    // arithmetic of the loads behind the barrier, which costs the step about 3 % - paid on one
    // step in kPollSteps instead of on all of them. The last two steps have nothing left to
    // load (`loading` kNoTile), the last one nothing to read ahead either (`reading_ahead`
    // false): after its barrier no wave touches the tile buffers any more. False: the
    // work-group has to leave.
    auto step = [&](int t, auto polling, auto loading, auto reading_ahead) -> bool {
        constexpr bool kPoll = decltype(polling)::value;
        constexpr int kLoad = decltype(loading)::value;
        constexpr bool kReadAhead = decltype(reading_ahead)::value;
        constexpr bool kMask = kFit != Fit::kExact && !kReadAhead;
        const int cur = t & 1;
        // Wave 0 asks for the preempt word here, with a vector load that is on its way during
        // the first slice, and looks at it just before the barrier: no wave ever waits for the
        // word alone (a scalar load at the barrier made wave 0 wait for the uncached round trip
        // and for all of its LDS reads while the other seven waves stood at the barrier).
        uint32_t polled = 0;
        if (kPoll && wave == 0) polled = xguard_read_flag_begin(xguard_flag_copy(g, blockIdx.x));

        // First slice: one read next to each of the first MFMAs, so that all have arrived by its end.
        if (kMask) mask_behind_k(0);
        XS_PIN;
#pragma unroll
        for (int n = 0; n < kMfmas; ++n) {
            mfma(0, n);
            if (n < kReads) read_frag(cur, 1, n);
            XS_PIN;
        }
        if (kMask) mask_behind_k(1);

        if (kPoll && wave == 0) {
            const bool current = xguard_read_flag_end(polled) == g.epoch;
            if (lane == 0) {
                if (!current) xguard_note_flush(g);
                guard_word = current ? 1u : 0u;
            }
        }
        XS_WAIT_GLOBAL_LOADS; // this wave's part of tile t + 1 has landed
        __syncthreads();      // tile t + 1 is complete, nobody reads buffer cur any more
        if (kPoll) {
            if (*(LdsVolatileWord *)&guard_word == 0) return false; // the whole group leaves together; nothing was written, no load is in flight
        }

        // Second slice: next to its MFMAs the first fragments of tile t + 1, one to every second MFMA,
        // and the loads of tile t + 2 into the buffer that has just become free.
        XS_PIN;
#pragma unroll
        for (int n = 0; n < kMfmas; ++n) {
            mfma(1, n);
            if (kReadAhead && n % 2 == 0 && n / 2 < kReads) read_frag(cur ^ 1, 0, n / 2);
            if (n % kLoadEvery == kLoadEvery - 1 && n / kLoadEvery < kLoads) {
                if constexpr (kLoad == kAnyButLast) load_piece(cur, t + 2, n / kLoadEvery, false);
                if constexpr (kLoad == kTheLast) load_piece(cur, t + 2, n / kLoadEvery, true);
            }
            XS_PIN;
        }
        return true;
    };
    constexpr std::true_type yes {};
    constexpr std::false_type no {};
    constexpr std::integral_constant<int, kNoTile> no_tile {};
    constexpr std::integral_constant<int, kAnyButLast> any_but_last {};
    constexpr std::integral_constant<int, kTheLast> the_last {};

    // steps that request a tile (kExact: the last one is like the others)
    const int main_steps = steps - 2 - (kFit == Fit::kExact ? 0 : 1);
    if constexpr (!kGuard) {
        for (int t = 0; t < main_steps; ++t) step(t, no, any_but_last, yes);
    } else {
        for (int t0 = 0; t0 < main_steps; t0 += kPollSteps) {
            const int last = min(t0 + kPollSteps, main_steps) - 1;
            for (int t = t0; t < last; ++t) step(t, no, any_but_last, yes);
            if (!step(last, yes, any_but_last, yes)) return;
        }
    }
    if constexpr (kFit != Fit::kExact) {
        if (steps > 2) step(steps - 3, no, the_last, yes);
    }
    if (steps >= 2) step(steps - 2, no, no_tile, yes);
    step(steps - 1, no, no_tile, no);

    // Write-out. A lane holds four consecutive rows of one column of each 16x16 block, so storing
    // from the accumulators would mean 2-byte stores to four different rows. Instead every wave
    // turns its strips of 32 rows x 64 columns over in LDS, in an area of its own inside the
    // tile buffers (nobody reads those any more, and nothing is on its way into them): a block's
    // four rows of one column go in as ONE 64-bit store (the strip is kept column-major, a column
    // padded from 64 to 80 bytes so that the sixteen columns of a store fall into different
    // banks), and the transposing read
    // brings it back out row-major: pointed at four rows of columns 8 q + j (lane 4 j + q of
    // every 16), it hands lane l row (l & 3) of columns 8 (l >> 2) + 0..3; a second read four
    // columns further completes 16 bytes per lane, and 8 rows x 128 bytes leave per store.
    constexpr int kStripColumnBytes = 64 + 16;
    constexpr int kStripBytes = 64 * kStripColumnBytes;
    static_assert(2 * (kABytes + kBBytes) >= kWaves * kStripBytes, "the tile buffers hold one strip per wave");
    uint8_t *const strip = As0 + wave * kStripBytes;
    const uint32_t l16 = lane & 15, patch = lane >> 4;   // a patch: 4 rows x 32 columns per 16 lanes
    const uint32_t put_at = l16 * kStripColumnBytes + 4 * patch * 2;
    const bool whole = WholeRowPieces(C, N);
    const uint32_t get_row = 4 * (patch >> 1), get_col = 32 * (patch & 1);
    const uint32_t get_at = (get_col + 8 * (l16 & 3) + (l16 >> 2)) * kStripColumnBytes + get_row * 2;
#pragma unroll
    for (int s = 0; s < kBlocksM / 2; ++s) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int j = 0; j < kBlocksN; ++j) {
                const f32x4 v = acc[2 * s + half][j];
                *(u32x2 *)(strip + 16 * j * kStripColumnBytes + put_at + 16 * half * 2) =
                    u32x2 { f32x2_to_bf16x2_rne(v.x, v.y), f32x2_to_bf16x2_rne(v.z, v.w) };
            }
        }
        const size_t row0 = m0 + 16 * kBlocksM * wm + 32 * s;
        const size_t col0 = n0 + 64 * wn + get_col + 8 * (l16 >> 2);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint8_t *p = strip + get_at + 8 * q * 2;
            const s16x4 left = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)p);
            const s16x4 right = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)(p + 4 * kStripColumnBytes));
            const s16x8 row = __builtin_shufflevector(left, right, 0, 1, 2, 3, 4, 5, 6, 7);
            // (non-temporal: C is written once and not read again; left in L2 it pushes out A and B panels
            // that the XCD's other tiles still need: 1 % of the kernel)
            StoreEight<kFit>(C, row0 + 8 * q + get_row + (l16 & 3), col0, M, N, whole, row);
        }
    }

    if (kGuard) guard.Commit();
}

template <bool kGuard, Fit kFit, int kTileM, int kTileN, int kWavesM, int kWavesN>
__global__ __launch_bounds__(64 * kWavesM * kWavesN, 2 /* waves per SIMD: no accumulators move between AGPRs and VGPRs */)
void GemmBf16Kernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                    uint16_t *__restrict__ C, int M, int N, int K, int lda, int ldb, XGuardArgs g)
{
    GemmBf16Body<kGuard, kFit, kTileM, kTileN, kWavesM, kWavesN>(A, B, C, M, N, K, lda, ldb, g);
}


// ---- smaller tiles, any shape ------------------------------------------------------------
//
// 128 x 128 or 64 x 64 tiles of C, four waves in a 2 x 2 grid, for outputs of too few large
// tiles to fill the device and for every shape the large tiles do not fit. One such work-group
// sits on a compute unit with one wave per SIMD, so nothing but its own instruction stream
// hides latencies; what bounds it is the round trip to memory (0.8-1 us, several K steps) and
// then LDS bandwidth (a 64 x 64 wave tile reads 16 KiB per 16 MFMAs of 32 cycles). Hence:
//   - kStages tiles of A and B are in LDS or on their way (4 x 32 KiB or 4 x 16 KiB), and the
//     waits count loads instead of draining them: s_waitcnt vmcnt leaves the newer tiles in
//     flight;
//   - the fragments of a WHOLE step are read from LDS into registers one step ahead, so a step
//     is one wait, one barrier and then MFMAs with an LDS read and a load next to each: the
//     buffer of tile t is free as soon as step t begins, and no MFMA waits for LDS.
// Layouts in LDS are of the kind of the kernel above, for fragments of 32x32x16 and with swizzles of their own:
//   A tile [kTile rows][64 k], two rows to a 256-byte line of sixteen slots of 16 bytes,
//          slot = ((row & 1) * 8 + k / 8) ^ (line & 15)
//   B tile as it sits in memory, [64 k][kTile cols], in granules of 64 bytes, granule = (col / 32) ^ (k & 3), on
//          tiles of 64, with two granules to a row, ^ ((k >> 1) & 1)
// The order of the additions is the same; the results are bit-identical.
//
// Measured, per guarded command in a stream of them (before: 128 x 128 tiles with one tile of
// lead, or a bounds-checked kernel of 64 x 64 tiles for what is not a multiple of the tiles):
//   1024^3            10.8 -> 5.8 us (64 x 64: 256 work-groups instead of 64)
//   2048^3            23.7 -> 17.8 us = 0.96 PFLOP/s
//   2000^3            86.5 -> 21.8 us      2000 x 1999 x 2047   254 -> 28.5 us
//   128 x 128 x 8192  76.0 -> 19.7 us      4097 x 4095 x 4097   2122 -> 243 us

/// What a K step does besides its MFMAs (see GemmDeepBody).
enum LoadKind { kNothing, kWholeTile, kLastTile };
template <int kLoad_, int kPut_, bool kRead_, int kNewer_>
struct Step
{
    static constexpr int kLoad = kLoad_;     // request a tile
    static constexpr int kPut = kPut_;       // kUnaligned: store a tile that has arrived to LDS
    static constexpr bool kRead = kRead_;    // read the next tile's fragments
    static constexpr int kNewer = kNewer_;   // tiles in flight behind the one waited for
};

/// s_waitcnt vmcnt(n) lgkmcnt(0)
template <int kVm>
__device__ __forceinline__ void WaitLoadsAndLds()
{
    static_assert(kVm >= 0 && kVm < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt((kVm & 15) | (7 << 4) | ((kVm >> 4) << 14));
}

/// s_waitcnt as above with at most `newer` tiles of kLoads loads in flight (`newer` is uniform, at most kMost).
template <int kMost, int kLoads>
__device__ __forceinline__ void WaitNewer(int newer)
{
    if constexpr (kMost == 0) WaitLoadsAndLds<0>();
    else if (newer >= kMost) WaitLoadsAndLds<kMost * kLoads>();
    else WaitNewer<kMost - 1, kLoads>(newer);
}

/// K of every tile divided among `parts` work-groups, `steps` K steps each (the last of them what is left).
/// Outputs of few tiles leave most of the device idle, and a step is bound by what one compute unit loads and
/// multiplies. A group stores its sums to partials (a tile of floats per group, as they lie in the
/// registers) and draws a ticket of its tile; who draws the last one adds up the parts in their order,
/// whichever group it is, so that the result does not depend on who came when, and writes C. A
/// ticket word holds the number of the launch that last used it (they ascend) above the tickets drawn.
/// Partial sums and tickets are of use to their own launch only: a tile has ONE byte in the progress map, tagged by who
/// has written it, and a replay does all parts of the other tiles anew. What other launches do to the
/// buffer between a flush and the replay does not matter.
/// Without memory for all this (or under capture) one work-group does the parts of a tile one after the other and
/// adds up their sums in the same order (Sum::kInTurn: only `steps` is used). In a graph's replay 128 x 128 x 8192 takes
/// 20.0 us that way and 16.6 in one go, 500 x 499 x 4095 22.2 both ways.
/// Plain launches and split ones, us per command: see QuickestPlan().
enum class Sum { kOneGo, kSplit, kInTurn };
struct SplitK
{
    float *partials;
    unsigned long long *tickets;   // one per tile
    unsigned long long launch;     // its number (SharedScratch)
    uint32_t parts, steps;
};
constexpr int kTicketBits = 24;    // below the launch's number
constexpr uint32_t kMaxSplitTiles = 256;
constexpr int kLeastLastSteps = 5; // of the last part
static_assert(kMaxSplitTiles <= SharedScratch::kTicketWords, "a ticket per tile");

template <bool kGuard, Fit kFit, int kTile, int kStages, Sum kSum>
__device__ __forceinline__
void GemmDeepBody(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                  uint16_t *__restrict__ C, int M, int N, int K, int lda, int ldb, const XGuardArgs &g, const SplitK &split)
{
    constexpr bool kSplit = kSum == Sum::kSplit;
    constexpr bool kDirect = kFit != Fit::kUnaligned;      // loads go straight into LDS
    constexpr int kWaves = 4;
    constexpr int kBlocks = kTile / 64;                    // 32x32 blocks per wave in each direction
    constexpr int kSlices = kStepK / 16;
    constexpr int kMfmas = kSlices * kBlocks * kBlocks;    // per wave and step
    constexpr int kFrags = kSlices * kBlocks;              // fragments of A (and of B) per wave and step
    constexpr int kTileBytes = kTile * kStepK * 2;         // A or B tile in LDS
    constexpr int kHalfLoads = kTileBytes / 1024 / kWaves; // 1 KiB loads per wave of one of them
    constexpr int kLoads = 2 * kHalfLoads;
    constexpr int kRegTiles = 2;                           // kUnaligned: tiles in flight in registers
    constexpr int kBuffers = kDirect ? kStages : 2;
    constexpr int kBRowBytes = kTile * 2;
    constexpr int kBSlotsPerRow = kBRowBytes / 16;
    constexpr int kBRowsPerLoad = 64 / kBSlotsPerRow;
    static_assert(2 * kFrags % kMfmas == 0 || 2 * kFrags <= kMfmas, "reads pair up with the MFMAs of a step");
    static_assert((kStages & (kStages - 1)) == 0 && kStages >= 4, "stages are numbered modulo a power of two");
    // one LDS object (see above): the tiles, then two slots for the preempt word, one for the `flushed` word and the
    // guard's own word
    constexpr int kFlagAt = 2 * kBuffers * kTileBytes;
    constexpr int kFlushedSlot = 2;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kFlagAt + 3 * 256 + 16];
    uint32_t &guard_word = *(uint32_t *)(lds + kFlagAt + 3 * 256);
    uint8_t *const As0 = lds;
    uint8_t *const Bs0 = lds + kBuffers * kTileBytes;

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t wm = wave >> 1, wn = wave & 1;

    uint32_t tm, tn;
    const uint32_t tiles_m = ((uint32_t)M + kTile - 1) / kTile, tiles_n = ((uint32_t)N + kTile - 1) / kTile;
    const uint32_t tiles = tiles_m * tiles_n, work = WorkOf(blockIdx.x, kSplit ? tiles * split.parts : tiles);
    const uint32_t part = kSplit ? work / tiles : 0, tile = kSplit ? work - part * tiles : work;   // (neighbours share A and B, parts share nothing)
    TileAt(tile, tiles_m, tiles_n, tm, tn);
    const size_t m0 = (size_t)tm * kTile, n0 = (size_t)tn * kTile;
    const int all_steps = kFit == Fit::kExact ? K / kStepK : (K + kStepK - 1) / kStepK;
    const int first_step = kSplit ? (int)(part * split.steps) : 0;
    const int steps = kSplit ? min((int)split.steps, all_steps - first_step) : all_steps;
    // K values of the last step
    const int rest = kFit == Fit::kExact || (kSplit && first_step + steps < all_steps) ? kStepK : K - (all_steps - 1) * kStepK;

    // ---- what each lane fetches for its LDS slot (see the layouts): byte offsets from the tile's first element ----
    uint32_t off[kLoads];
    uint32_t k_of[kLoads];                                 // the piece's first k within the step
#pragma unroll
    for (int i = 0; i < kHalfLoads; ++i) {
        const uint32_t q = wave * kHalfLoads + i;
        const uint32_t line = 4 * q + (lane >> 4);
        const uint32_t piece = (lane & 15) ^ (line & 15);
        uint32_t row = 2 * line + (piece >> 3);
        const uint32_t kc = piece & 7;
        if (kFit != Fit::kExact && m0 + row >= (size_t)M) row = (uint32_t)((size_t)M - 1 - m0);
        off[i] = (row * (uint32_t)lda + kc * 8) * 2;
        k_of[i] = kc * 8;
    }
#pragma unroll
    for (int i = 0; i < kHalfLoads; ++i) {
        const uint32_t q = wave * kHalfLoads + i;
        const uint32_t k = kBRowsPerLoad * q + lane / kBSlotsPerRow;
        const uint32_t slot = lane % kBSlotsPerRow;
        const uint32_t swz = kTile == 64 ? (k >> 1) & 1 : k & 3;
        uint32_t col = ((slot >> 2) ^ swz) * 32 + (slot & 3) * 8;
        if (kFit != Fit::kExact && n0 + col >= (size_t)N) col = 0;
        off[kHalfLoads + i] = (k * (uint32_t)ldb + col) * 2;
        k_of[kHalfLoads + i] = k;
    }
    const uint16_t *const a_tile = A + m0 * (size_t)lda + (size_t)first_step * kStepK;     // + kStepK columns per step
    const uint16_t *const b_tile = B + n0 + (size_t)first_step * kStepK * (size_t)ldb;     // + kStepK rows per step

    // Offset of piece idx in the last step: pieces behind K come from k = 0 of the step instead.
    auto last_off = [&](int idx) -> uint32_t {
        if (kFit == Fit::kExact || k_of[idx] < (uint32_t)rest) return off[idx];
        return idx < kHalfLoads ? off[idx] - k_of[idx] * 2 : off[idx] - k_of[idx] * (uint32_t)ldb * 2;
    };
    auto load_direct = [&](int step, int idx, uint32_t at) {
        const int buf = step & (kBuffers - 1);
        if (idx < kHalfLoads) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(a_tile + (size_t)step * kStepK), 0, 0x7fffffff, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)(As0 + buf * kTileBytes + (wave * kHalfLoads + idx) * 1024), 16, at, 0, 0, 0);
        } else {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)(b_tile + (size_t)step * kStepK * ldb), 0, 0x7fffffff, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)(Bs0 + buf * kTileBytes + (wave * kHalfLoads + idx - kHalfLoads) * 1024), 16, at, 0, 0, 0);
        }
    };
    // kUnaligned: the pieces of kRegTiles tiles on their way through registers
    u32x4 held[kDirect ? 1 : kRegTiles][kDirect ? 1 : kLoads];
    auto load_held = [&](int set, int step, int idx) {
        const uint8_t *base = idx < kHalfLoads ? (const uint8_t *)(a_tile + (size_t)step * kStepK)
                                               : (const uint8_t *)(b_tile + (size_t)step * kStepK * ldb);
        held[set][idx] = *(const u32x4_any *)(base + off[idx]);
    };
    // The last step's pieces: one that would reach behind the matrix is fetched from its last 16 bytes
    // instead, and shifted into place when it is put into LDS (not here: the shift would wait for the
    // load); what is then missing lies behind K or in columns behind N.
    auto last_piece = [&](int step, int idx, uint32_t &shift) -> const uint8_t * {
        const uint8_t *base = idx < kHalfLoads ? (const uint8_t *)(a_tile + (size_t)step * kStepK)
                                               : (const uint8_t *)(b_tile + (size_t)step * kStepK * ldb);
        const uint8_t *const end = idx < kHalfLoads ? (const uint8_t *)(A + (size_t)M * K) : (const uint8_t *)(B + (size_t)K * N);
        const uint8_t *const p = base + last_off(idx);
        const uint8_t *const inside = p + 16 <= end ? p : end - 16;
        shift = (uint32_t)(p - inside);
        return inside;
    };
    auto load_held_last = [&](int set, int step, int idx) {
        uint32_t shift;
        held[set][idx] = *(const u32x4_any *)last_piece(step, idx, shift);
    };
    auto put_held = [&](int set, int step, int idx, bool last) {
        const int buf = step & (kBuffers - 1);
        uint8_t *const at = idx < kHalfLoads ? As0 + buf * kTileBytes + (wave * kHalfLoads + idx) * 1024
                                             : Bs0 + buf * kTileBytes + (wave * kHalfLoads + idx - kHalfLoads) * 1024;
        uint32_t shift = 0;
        if (last) (void)last_piece(step, idx, shift);
        *(u32x4 *)(at + lane * 16) = last ? ShiftDownBytes(held[set][idx], shift) : held[set][idx];
    };

    // ---- LDS -> fragments: the same layouts the other way round ----
    const uint32_t a_row0 = 32 * kBlocks * wm + (lane & 31);
    const uint32_t a_line = a_row0 >> 1;
    const uint32_t a_base = a_line * 256 + (((((lane & 1) << 3) | (lane >> 5)) ^ (a_line & 15)) << 4);
    const uint32_t b_row = 8 * (lane >> 5) + ((lane & 15) >> 2);
    const uint32_t b_swz = kTile == 64 ? (b_row >> 1) & 1 : b_row & 3;
    const uint32_t b_base = b_row * kBRowBytes + (((kBlocks * wn) ^ b_swz) << 6) + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
    bf16x8 fa[2][kFrags], fb[2][kFrags];                   // [parity of the step][slice * kBlocks + block]
    // Fragment unit n of tile `step` into set `set`: A and B of a slice next to each other.
    auto read_unit = [&](int set, int step, int n) {
        const int buf = step & (kBuffers - 1);
        const int ks = n / (2 * kBlocks), r = n % (2 * kBlocks);
        if (r < kBlocks) {
            fa[set][ks * kBlocks + r] = *(const bf16x8 *)(As0 + buf * kTileBytes + (a_base ^ (ks << 5)) + r * 4096);
        } else {
            const int j = r - kBlocks;
            const uint8_t *p = Bs0 + buf * kTileBytes + ks * 16 * kBRowBytes + (b_base ^ (j << 6));
            const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)p);
            const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)(p + 4 * kBRowBytes));
            fb[set][ks * kBlocks + j] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    };

    f32x16 acc[kBlocks][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto mfma = [&](int set, int n) {
        const int ks = n / (kBlocks * kBlocks), i = n / kBlocks % kBlocks, j = n % kBlocks;
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[set][ks * kBlocks + i], fb[set][ks * kBlocks + j], acc[i][j], 0, 0, 0);
    };
    // kInTurn: the sums of the parts that have ended, of none -0: adding to that changes nothing. (Parts are of an even number
    // of steps, and the last one of at least kLeastLastSteps: the others end between two pairs of steps of the main loop.)
    f32x16 ended[kSum == Sum::kInTurn ? kBlocks : 1][kSum == Sum::kInTurn ? kBlocks : 1];
    if constexpr (kSum == Sum::kInTurn) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) ended[i][j][r] = -0.f;
    }
    auto add_ended_part = [&]() {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    ended[i][j][r] += acc[i][j][r];
                    acc[i][j][r] = 0.f;
                }
    };
    // A lane's fragment of slice ks holds k = 16 ks + 8 (lane / 32) + 0..7 of the step, for A and
    // for B alike: everything from `rest` on becomes zero.
    auto mask_behind_k = [&](int set) {
#pragma unroll
        for (int ks = 0; ks < kSlices; ++ks) {
            const int valid = rest - (16 * ks + 8 * (int)(lane >> 5));
            u32x4 m;
#pragma unroll
            for (int d = 0; d < 4; ++d) m[d] = valid >= 2 * d + 2 ? 0xFFFFFFFFu : valid == 2 * d + 1 ? 0xFFFFu : 0u;
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) {
                fa[set][ks * kBlocks + i] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fa[set][ks * kBlocks + i]) & m);
                fb[set][ks * kBlocks + i] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, fb[set][ks * kBlocks + i]) & m);
            }
        }
    };
#define XS_BARRIER do { asm volatile("" ::: "memory"); XS_PIN; __builtin_amdgcn_s_barrier(); XS_PIN; asm volatile("" ::: "memory"); } while (0)

    // ---- prologue: the first tiles on their way, the guard's words in front of them ----
    // The words travel like a tile: wave 0 has them loaded into LDS (one wave-wide load each, in order with
    // the tiles'), and every wave reads them there once tile 0 has been waited for in front of a
    // barrier. (A load into a register would have to be waited for with all tiles requested behind it
    // as far as the compiler can tell; scalar loads are two more round trips, and the decision a barrier of its own.)
    // A replay also looks at its byte of the progress map, the ordinary way.
    const XGuardBlock guard(g, kSplit ? tile : blockIdx.x, &guard_word);
    auto request_word = [&](const uint32_t *word, int slot) {
        if (wave == 0) {
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)word, 0, 4, 0x00020000);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (LdsVoid *)(lds + kFlagAt + slot * 256), 4, 0, 0, 0, 0x11 /* sc0 sc1: system scope */);
        }
    };
    auto word_of = [&](int slot) -> uint32_t {
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)*(LdsVolatileWord *)(lds + kFlagAt + slot * 256));
    };
    auto request_flag = [&](int slot) { request_word(xguard_flag_copy(g, blockIdx.x), slot); };
    auto flag_is_current = [&](int slot) -> bool { return word_of(slot) == g.epoch; };
    const bool by_words = kGuard && !xguard_inert(g) && !g.resume && g.flushed != nullptr;
    if (kGuard) {
        if (by_words) {
            request_flag(1);
            request_word(g.flushed, kFlushedSlot);
        } else if (!guard.Enter()) {
            return;
        }
    }
    // Waits until tile t has landed, i.e. all but the `newer` tiles requested behind it.
    auto wait_tile = [&](int newer) { WaitNewer<kStages - 1, kLoads>(newer); };
    // Tiles 0, 1, .. on their way, tile 0 (kUnaligned: and 1) waited for. `many`: at least kTail steps, none of
    // these tiles is the last, and there is no branch between loads. (With branches the compiler loses
    // count of the loads in flight behind them: at the head of the main loop it then waited for all of them but one,
    // and through registers a step in four took the round trip to memory.)
    auto request_first = [&](auto many) {
        constexpr bool kMany = decltype(many)::value;
        constexpr int kAhead = kDirect ? kStages : kRegTiles;
#pragma unroll
        for (int t = 0; t < kAhead; ++t) {
            if (!kMany && t >= steps) break;
#pragma unroll
            for (int idx = 0; idx < kLoads; ++idx) {
                if constexpr (kDirect) load_direct(t, idx, !kMany && t == steps - 1 ? last_off(idx) : off[idx]);
                else if (!kMany && t == steps - 1) load_held_last(t, t, idx);
                else load_held(t, t, idx);
                if constexpr (kMany && !kDirect) XS_PIN;   // (in this order, which the waits count on)
            }
        }
        if constexpr (kDirect) {
            if constexpr (kMany) WaitLoadsAndLds<(kStages - 1) * kLoads>();
            else wait_tile(min(kStages, steps) - 1);
        } else {
            // tile 0, then tile 1, into their LDS buffers; the next ones into the registers they leave
#pragma unroll
            for (int t = 0; t < kRegTiles; ++t) {
                if (kMany || t < steps) {
#pragma unroll
                    for (int idx = 0; idx < kLoads; ++idx) put_held(t, t, idx, !kMany && t == steps - 1);
                }
                const int next = t + kRegTiles;
                if (kMany || next < steps - 1) {
#pragma unroll
                    for (int idx = 0; idx < kLoads; ++idx) {
                        load_held(t, next, idx);
                        if constexpr (kMany) XS_PIN;
                    }
                } else if (next == steps - 1) {
#pragma unroll
                    for (int idx = 0; idx < kLoads; ++idx) load_held_last(t, next, idx);
                }
            }
            static_assert(kDirect || kRegTiles == kBuffers, "tiles 0 .. kRegTiles - 1 each have a buffer");
            __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the stores to LDS are done (tile 0 has come through registers, and the guard's words before it)
        }
    };
    // The barrier that tile 0 is complete behind, and the guard's decision; false: the group has to leave.
    auto enter = [&]() -> bool {
        XS_BARRIER;
        if (kGuard && by_words) {
            const XGuardVerdict v = xguard_entry_verdict(word_of(1), word_of(kFlushedSlot), g.epoch, 0, 0, 0, g.gen);
            if (!v.run) {
                XS_WAIT_GLOBAL_LOADS; // nothing may still be on its way into LDS when the group is gone
                if (v.note_flush && tid == 0) xguard_note_flush(g);
                return false;
            }
        }
        return true;
    };

    // Later looks at the preempt word are the same: requested into LDS, and kPollSteps steps later, when
    // that load has landed because loads requested behind it have been waited for in front of a barrier,
    // read there by every wave. (A scalar load would have to be waited for with all LDS reads.) Two slots
    // in turn (the one of the entry is the second): between two writes of one slot lie the barriers of
    // eight steps and one look at it.

    // One step. Tile t + 1 is waited for (kNewer tiles requested behind it stay in flight), then
    // come the MFMAs on the fragments of tile t, next to them the fragment reads of tile t + 1 and
    // the loads of the tile that goes into the buffer that has just become free. `what` says what
    // is left to do besides the MFMAs; all of it is known where a step is written down, for the
    // last steps too: a branch in a step would make its MFMAs wait for its reads.
    auto step = [&](int t, auto parity, auto what) {
        constexpr int p = decltype(parity)::value;
        using Do = decltype(what);
        XS_PIN;
        if constexpr (kDirect) WaitLoadsAndLds<Do::kNewer * kLoads>();
        else __builtin_amdgcn_s_waitcnt(0xC07F);
        XS_BARRIER;
        if constexpr (kFit != Fit::kExact && !Do::kRead) {
            if (rest != kStepK) mask_behind_k(p);
        }
#pragma unroll
        for (int n = 0; n < kMfmas; ++n) {
            mfma(p, n);
            constexpr int kReads = 2 * kFrags >= kMfmas ? 2 * kFrags / kMfmas : 1;
#pragma unroll
            for (int r = n * kReads; Do::kRead && r < (n + 1) * kReads && r < 2 * kFrags; ++r) read_unit(p ^ 1, t + 1, r);
#pragma unroll
            for (int idx = n * kLoads / kMfmas; idx < (n + 1) * kLoads / kMfmas; ++idx) {
                if constexpr (kDirect) {
                    if constexpr (Do::kLoad == kWholeTile) load_direct(t + kStages, idx, off[idx]);
                    if constexpr (Do::kLoad == kLastTile) load_direct(t + kStages, idx, last_off(idx));
                } else {
                    if constexpr (Do::kPut != kNothing) put_held(p, t + 2, idx, Do::kPut == kLastTile);
                    if constexpr (Do::kLoad == kWholeTile) load_held(p, t + 2 + kRegTiles, idx);
                    if constexpr (Do::kLoad == kLastTile) load_held_last(p, t + 2 + kRegTiles, idx);
                }
            }
            XS_PIN;
        }
    };
    constexpr std::integral_constant<int, 0> even {};
    constexpr std::integral_constant<int, 1> odd {};
    using Main = Step<kWholeTile, kWholeTile, true, kStages - 2>;

    // The main steps load whole tiles; the kTail steps behind them load the last tile (kExact: it
    // is like the others) or nothing, and the last reads no fragments.
    constexpr int kTail = kDirect ? (kFit == Fit::kExact ? kStages : kStages + 1) : 3 + kRegTiles;
    static_assert(kTail <= kLeastLastSteps, "parts end in the main loop");
    if (steps >= kTail) {
        static_assert(kTail > (kDirect ? kStages : 2 * kRegTiles) || kFit == Fit::kExact, "request_first() meets no last tile");
        request_first(std::true_type {});
        if (!enter()) return;
        const int main_steps = steps - kTail;
        int t = 0;
#pragma unroll
        for (int n = 0; n < 2 * kFrags; ++n) read_unit(0, 0, n);
        static_assert(kPollSteps == 4 && kStages <= kPollSteps + 2, "a request has landed by the last barrier in front of its look");
        uint32_t slot = 0;
        if (kGuard && main_steps >= kPollSteps) request_flag(0);
        // main steps up to `end`, in pairs; false: the group has to leave
        auto steps_to = [&](int end) -> bool {
            if constexpr (kGuard) {
                for (; t + kPollSteps <= end; t += kPollSteps) {
                    step(t, even, Main {}); step(t + 1, odd, Main {});
                    step(t + 2, even, Main {}); step(t + 3, odd, Main {});
                    if (!flag_is_current(slot)) {   // the same word in every wave: the group leaves together
                        XS_WAIT_GLOBAL_LOADS;
                        if (tid == 0) xguard_note_flush(g);
                        return false;
                    }
                    slot ^= 1;
                    request_flag(slot);
                }
            }
            for (; t + 2 <= end; t += 2) { step(t, even, Main {}); step(t + 1, odd, Main {}); }
            return true;
        };
        if constexpr (kSum == Sum::kInTurn) {
            const int part = (int)split.steps;
            for (int end = part; ; end += part) {
                if (!steps_to(min(end, main_steps))) return;
                if (t != end) break;   // in the last part
                add_ended_part();
            }
        } else {
            if (!steps_to(main_steps)) return;
        }
        auto tail = [&](auto first_parity) {
            constexpr int p = decltype(first_parity)::value;
            auto at = [&]<int j>(std::integral_constant<int, j>) {
                constexpr int left = kTail - 1 - j;                              // steps behind this one
                constexpr bool loads_last = kFit != Fit::kExact && j == 0;
                constexpr int newer = left - 1 < 0 ? 0 : left - 1 < kStages - 2 ? left - 1 : kStages - 2;
                using Do = Step<loads_last ? kLastTile : kNothing, (left > 2 ? kWholeTile : left == 2 ? kLastTile : kNothing), (left >= 1), newer>;
                step(main_steps + j, std::integral_constant<int, (p + j) & 1> {}, Do {});
            };
            [&]<int... j>(std::integer_sequence<int, j...>) { (at(std::integral_constant<int, j> {}), ...); }(std::make_integer_sequence<int, kTail> {});
        };
        if (t < main_steps) {
            step(t, even, Main {});
            tail(odd);
        } else {
            tail(even);
        }
    } else {
        // K of a few steps: everything is on its way (or here) already, and the fragments are
        // read in front of their MFMAs.
        request_first(std::false_type {});
        if (!enter()) return;
        if constexpr (kDirect) WaitLoadsAndLds<0>();
        XS_BARRIER;
        for (int t = 0; t < steps; ++t) {
#pragma unroll
            for (int n = 0; n < 2 * kFrags; ++n) read_unit(0, t, n);
            if (kFit != Fit::kExact && t == steps - 1) mask_behind_k(0);
#pragma unroll
            for (int n = 0; n < kMfmas; ++n) mfma(0, n);
            if constexpr (!kDirect) {
                // the buffer just read takes the tile after the next one
                WaitLoadsAndLds<0>();
                XS_BARRIER;
#pragma unroll
                for (int idx = 0; idx < kLoads; ++idx) {
                    if (t + 2 < steps) { if (t & 1) put_held(1, t + 2, idx, t + 2 == steps - 1); else put_held(0, t + 2, idx, t + 2 == steps - 1); }
                }
                WaitLoadsAndLds<0>();
                XS_BARRIER;
            }
        }
        XS_PIN;
        WaitLoadsAndLds<0>();
        XS_BARRIER;
    }
    if (kGuard) XS_WAIT_GLOBAL_LOADS;                      // the last look at the preempt word that nobody took

    if constexpr (kSplit) {
        // Partial sums go past the L2 of the group's XCD (system-coherent accesses of device scope, sc1) and are read the same
        // way: they have arrived when the wave's stores have, and no L2 is written back or
        // invalidated (with release fences, 256 groups took 20 us longer).
        constexpr int kThreads = 64 * kWaves, kDeviceScope = 0x10;
        constexpr int kPieces = kBlocks * kBlocks * 4;
        constexpr int kPartBytes = kTile * kTile * 4;
        constexpr int kUnroll = kTile == kTinyTile ? 4 : 1;   // parts read at a time: as many as fit into the registers
        const __amdgpu_buffer_rsrc_t parts = __builtin_amdgcn_make_buffer_rsrc((void *)(split.partials + (size_t)tile * split.parts * (kTile * kTile)), 0,
                                                                               (int)(split.parts * kPartBytes), 0x00020000);
        // (The part is in the resource and not in a scalar offset: with one the compiler lets the next instruction write
        // over the registers of a 16-byte store, as documented. Where it did so, in a form of eight waves,
        // lanes 12-15 of sixteen now and then stored the address that came next in place of their first value.)
        const __amdgpu_buffer_rsrc_t mine = __builtin_amdgcn_make_buffer_rsrc((void *)(split.partials + ((size_t)tile * split.parts + part) * (kTile * kTile)), 0,
                                                                              kPartBytes, 0x00020000);
#pragma unroll
        for (int n = 0; n < kPieces; ++n) {
            const f32x16 &v = acc[n / 4 / kBlocks][n / 4 % kBlocks];
            const f32x4 four = { v[n % 4 * 4], v[n % 4 * 4 + 1], v[n % 4 * 4 + 2], v[n % 4 * 4 + 3] };
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, four), mine, (n * kThreads + tid) * 16, 0, kDeviceScope);
        }
        XS_WAIT_GLOBAL_LOADS;   // (stores count as loads do)
        XS_BARRIER;
        if (tid == 0) {
            unsigned long long *const word = split.tickets + tile;
            (void)__hip_atomic_fetch_max(word, split.launch << kTicketBits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            const unsigned long long drawn = __hip_atomic_fetch_add(word, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            guard_word = ((uint32_t)drawn & ((1u << kTicketBits) - 1)) % split.parts == split.parts - 1 ? 1u : 0u;
        }
        __syncthreads();
        if (*(LdsVolatileWord *)&guard_word == 0) return;   // (not committed: a byte of the map stands for a tile)
        XS_PIN;
        f32x4 sum[kPieces];
        auto piece = [&](uint32_t p, int n) -> f32x4 {
            return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(parts, (n * kThreads + tid) * 16, p * kPartBytes, kDeviceScope));
        };
#pragma unroll
        for (int n = 0; n < kPieces; ++n) sum[n] = piece(0, n);
#pragma unroll kUnroll
        for (uint32_t p = 1; p < split.parts; ++p) {
#pragma unroll
            for (int n = 0; n < kPieces; ++n) sum[n] += piece(p, n);
        }
#pragma unroll
        for (int n = 0; n < kPieces; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[n / 4 / kBlocks][n / 4 % kBlocks][n % 4 * 4 + e] = sum[n][e];
    }

    if constexpr (kSum == Sum::kInTurn) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = ended[i][j][r] + acc[i][j][r];
    }

    // ---- write-out, as above: strips of 32 rows x 32 kBlocks columns turned over in LDS ----
    // (behind the last step's barrier nobody reads the tile buffers any more, and nothing is on
    // its way into them)
    constexpr int kStripColumnBytes = 64 + 8;
    constexpr int kStripBytes = 32 * kBlocks * kStripColumnBytes;
    static_assert(kBuffers * kTileBytes >= kWaves * kStripBytes, "the A buffers hold one strip per wave");
    uint8_t *const strip = As0 + wave * kStripBytes;
    const uint32_t put_at = (lane & 31) * kStripColumnBytes + 4 * (lane >> 5) * 2;
    const uint32_t l16 = lane & 15, patch = lane >> 4;     // a patch: 4 rows x 32 columns per 16 lanes
    constexpr int kRowsPerStore = 16 / kBlocks;
    const bool whole = WholeRowPieces(C, N);
    const uint32_t get_row = 4 * (patch / kBlocks), get_col = 32 * (patch % kBlocks);
    const uint32_t get_at = (get_col + 8 * (l16 & 3) + (l16 >> 2)) * kStripColumnBytes + get_row * 2;
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
#pragma unroll
            for (int run = 0; run < 4; ++run) {
                const uint32_t lo = f32x2_to_bf16x2_rne(acc[i][j][4 * run], acc[i][j][4 * run + 1]);
                const uint32_t hi = f32x2_to_bf16x2_rne(acc[i][j][4 * run + 2], acc[i][j][4 * run + 3]);
                *(u32x2 *)(strip + 32 * j * kStripColumnBytes + put_at + 8 * run * 2) = u32x2 { lo, hi };
            }
        }
        const size_t row0 = m0 + 32 * kBlocks * wm + 32 * i;
        const size_t col0 = n0 + 32 * kBlocks * wn + get_col + 8 * (l16 >> 2);
#pragma unroll
        for (int q = 0; q < 32 / kRowsPerStore; ++q) {
            const uint8_t *p = strip + get_at + kRowsPerStore * q * 2;
            const s16x4 left = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)p);
            const s16x4 right = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsS16x4 *)(p + 4 * kStripColumnBytes));
            const s16x8 eight = __builtin_shufflevector(left, right, 0, 1, 2, 3, 4, 5, 6, 7);
            const size_t row = row0 + kRowsPerStore * q + get_row + (l16 & 3);
            StoreEight<kFit>(C, row, col0, M, N, whole, eight);
        }
    }

    if (kGuard) guard.Commit();
}
#undef XS_BARRIER

template <bool kGuard, Fit kFit, int kTile, int kStages>
__global__ __launch_bounds__(256)
void GemmDeepKernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                    uint16_t *__restrict__ C, int M, int N, int K, int lda, int ldb, XGuardArgs g)
{
    GemmDeepBody<kGuard, kFit, kTile, kStages, Sum::kOneGo>(A, B, C, M, N, K, lda, ldb, g, SplitK {});
}

template <bool kGuard, Fit kFit, int kTile, int kStages, Sum kSum>
__global__ __launch_bounds__(256)
void GemmSplitKernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                     uint16_t *__restrict__ C, int M, int N, int K, int lda, int ldb, XGuardArgs g, SplitK split)
{
    GemmDeepBody<kGuard, kFit, kTile, kStages, kSum>(A, B, C, M, N, K, lda, ldb, g, split);
}

/// A queue's ticket words, before the first command that uses them.
__global__ __launch_bounds__(kMaxSplitTiles)
void ClearTicketsKernel(unsigned long long *tickets) { tickets[threadIdx.x] = 0; }


// Short K (ShortK() below), and what the kernels above do not take: fewer than eight columns or
// fewer than eight elements of A
// (less than one 16-byte piece to fetch), K or N above kMaxK (their 32-bit offsets). Any M, N, K >= 1,
// any alignment of the three matrices to two bytes. 64 x 64 tiles of C, four waves of one 32x32
// block each, K in steps of 32 (two slices of 16 through the same MFMA as above and in the same
// order; what lies beyond K is zero). Every load and store is checked against the matrix; a
// thread's eight neighbouring elements come as one 16-byte load where they lie inside the matrix
// and are aligned, one by one otherwise. The guard is at entry only: a tile is short.
// 10 KiB of LDS and few registers: many work-groups share a compute unit, and with short K, where
// a product is mostly the writing of C, one computes while the others write (us per command, the
// kernels above and this one: 7001 x 7003 x 32 89.3 -> 32.0, 2000 x 1999 x 16 9.4 -> 6.7,
// 4000 x 4008 x 32 13.7 -> 11.9, 300 x 301 x 8 5.2 -> 4.6).
constexpr int kAnyTile = 64;
constexpr int kAnyK = 32;

template <bool kGuard>
__global__ __launch_bounds__(256)
void GemmBf16AnyShapeKernel(const uint16_t *__restrict__ A, const uint16_t *__restrict__ B,
                            uint16_t *__restrict__ C, int M, int N, int K, uint32_t tiles_n, XGuardArgs g)
{
    // a row of 32 k values padded to 40: 80-byte rows, every 16-byte fragment aligned
    __shared__ __attribute__((aligned(16))) uint16_t a_rows[kAnyTile][kAnyK + 8];
    __shared__ __attribute__((aligned(16))) uint16_t b_cols[kAnyTile][kAnyK + 8];   // B transposed: [column][k]
    __shared__ uint32_t guard_word;

    const XGuardBlock guard(g, blockIdx.x, &guard_word);
    const XGuardEntry entry = kGuard ? guard.EnterBegin() : XGuardEntry {};

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const uint32_t wm = wave >> 1, wn = wave & 1;
    const size_t m0 = (size_t)(blockIdx.x / tiles_n) * kAnyTile, n0 = (size_t)(blockIdx.x % tiles_n) * kAnyTile;
    const size_t Ms = (size_t)M, Ns = (size_t)N, Ks = (size_t)K;

    // loads of a step: thread t takes A[m0 + t / 4][k0 + 8 (t % 4) + 0..7] and
    // B[k0 + t / 8][n0 + 8 (t % 8) + 0..7]
    const uint32_t a_row = tid >> 2, a_k = (tid & 3) * 8;
    const uint32_t b_k = tid >> 3, b_col = (tid & 7) * 8;
    union Eight { u32x4 v; uint16_t e[8]; };
    auto load_eight = [](const uint16_t *base, size_t first, size_t end, bool row_inside) {
        Eight r;
        r.v = u32x4 { 0, 0, 0, 0 };
        if (!row_inside || first >= end) return r;
        const uint16_t *p = base + first;
        if (first + 8 <= end && (((uintptr_t)p) & 15) == 0) {
            r.v = *(const u32x4 *)p;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) r.e[i] = first + i < end ? p[i] : (uint16_t)0;
        }
        return r;
    };
    auto load_a = [&](size_t k0) { return load_eight(A + (m0 + a_row) * Ks, k0 + a_k, Ks, m0 + a_row < Ms); };
    auto load_b = [&](size_t k0) { return load_eight(B + (k0 + b_k) * Ns, n0 + b_col, Ns, k0 + b_k < Ks); };

    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;

    Eight a = load_a(0), b = load_b(0);
    if (kGuard && !guard.EnterEnd(entry)) return;
    for (size_t k0 = 0; k0 < Ks; k0 += kAnyK) {
        __syncthreads();   // the fragments of the previous step have been read
        *(u32x4 *)&a_rows[a_row][a_k] = a.v;
#pragma unroll
        for (int i = 0; i < 8; ++i) b_cols[b_col + i][b_k] = b.e[i];
        __syncthreads();
        if (k0 + kAnyK < Ks) { a = load_a(k0 + kAnyK); b = load_b(k0 + kAnyK); }
        // lane l: A[row l % 32][k 8 (l / 32) + 0..7], B[k 8 (l / 32) + 0..7][column l % 32], per slice of 16
#pragma unroll
        for (int kk = 0; kk < kAnyK; kk += 16) {
            const bf16x8 fa = *(const bf16x8 *)&a_rows[32 * wm + (lane & 31)][kk + 8 * (lane >> 5)];
            const bf16x8 fb = *(const bf16x8 *)&b_cols[32 * wn + (lane & 31)][kk + 8 * (lane >> 5)];
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb, acc, 0, 0, 0);
        }
    }

    // accumulator 4 run + r of lane l: row 8 run + 4 (l / 32) + r, column l % 32 of the block
    const size_t col = n0 + 32 * wn + (lane & 31);
    if (col < Ns) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const size_t row = m0 + 32 * wm + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3);
            if (row < Ms) C[row * Ns + col] = (uint16_t)f32x2_to_bf16x2_rne(acc[i], 0.0f);
        }
    }
    if (kGuard) guard.Commit();
}

/// A matrix that is copied to rows on 16-byte boundaries: `rows` rows of `cols` elements, one after
/// the other from `from` on, to rows of `ld` (a multiple of 8) from `to` on. The elements of `to`
/// between cols and ld take whatever follows in memory: nothing depends on them (kEdges).
struct RowCopy
{
    const uint16_t *from;
    uint16_t *to;
    uint32_t rows, cols, ld;
    uint32_t groups;   // work-groups that copy it, 0: it stays where it is
};
constexpr uint32_t kCopyThreads = 256;
constexpr uint32_t kCopyPieces = 4;    // 16-byte pieces per thread, all on their way at once
inline uint32_t CopyGroups(uint64_t rows, uint64_t ld) { return (uint32_t)((rows * (ld / 8) + kCopyThreads * kCopyPieces - 1) / (kCopyThreads * kCopyPieces)); }

/// Copies A, B or both in one launch, for kernels whose loads go straight into LDS. Bound by memory: each
/// element is read and written once (the pieces are read at any multiple of two bytes, which memory
/// does not mind). The guard is at entry only: a group copies 16 KiB. A copy is of use to the launch behind it only (other
/// commands copy to the same place), so it has no progress byte, and a replay copies everything
/// anew unless all of the product's tiles have been written: tiles_done are their bytes, of the replay's map.
template <bool kGuard>
__global__ __launch_bounds__(kCopyThreads)
void CopyRowsKernel(RowCopy a, RowCopy b, const uint8_t *tiles_done, uint32_t tiles, XGuardArgs g)
{
    __shared__ uint32_t guard_word;
    const XGuardBlock guard(g, blockIdx.x, &guard_word);
    const XGuardEntry entry = kGuard ? guard.EnterBegin() : XGuardEntry {};
    if (kGuard && tiles_done != nullptr) {
        int missing = 0;
        for (uint32_t t = threadIdx.x; t < tiles; t += kCopyThreads) missing |= tiles_done[t] != (uint8_t)g.gen;
        if (__syncthreads_or(missing) == 0) return;
    }
    const bool second = blockIdx.x >= a.groups;
    const RowCopy &m = second ? b : a;
    const uint32_t pieces_per_row = m.ld / 8, pieces = m.rows * pieces_per_row;   // (at most 2^26: kMaxScratchBytes)
    const uint32_t first = (blockIdx.x - (second ? a.groups : 0)) * (kCopyThreads * kCopyPieces) + threadIdx.x;
    const size_t last = (size_t)m.rows * m.cols - 8;   // first element of the matrix's last 16 bytes
    u32x4 v[kCopyPieces];
    uint32_t d[kCopyPieces];
#pragma unroll
    for (uint32_t u = 0; u < kCopyPieces; ++u) {
        const uint32_t p = min(first + u * kCopyThreads, pieces - 1);
        const uint32_t row = p / pieces_per_row;
        const size_t at = (size_t)row * m.cols + (p - row * pieces_per_row) * 8;
        // a piece that would reach behind the matrix: its last 16 bytes, shifted into place
        const size_t inside = at < last ? at : last;
        v[u] = *(const u32x4_any *)(m.from + inside);
        d[u] = (uint32_t)(at - inside) * 2;
    }
    if (kGuard && !guard.EnterEnd(entry)) return;
#pragma unroll
    for (uint32_t u = 0; u < kCopyPieces; ++u) {
        const uint32_t p = first + u * kCopyThreads;
        if (p < pieces) *(u32x4 *)(m.to + (size_t)p * 8) = ShiftDownBytes(v[u], d[u]);   // rows of ld elements follow each other: piece p is p * 16 bytes on
    }
}

/// kTwoBuffers is GemmBf16Kernel, kFourStages GemmDeepKernel, kAnyShape GemmBf16AnyShapeKernel.
enum class Body { kTwoBuffers, kFourStages, kAnyShape };

/// A run of rows of C and how they are computed: which kernel, on tiles of which size, and what it
/// may assume about the matrices.
struct Part
{
    int first_row, rows;
    int tile;       // edge of a tile of C
    Fit fit;        // of kTwoBuffers and kFourStages
    Body body;
    uint64_t tiles; // work-groups, at least as many as bytes of the progress map (a byte for a tile)
    int tile_rows;  // rows of a tile: as many as `tile`, or with 256 columns and two buffers fewer
    Sum sum = Sum::kOneGo;                  // the others: kFourStages, one launch for all of C
    int split_parts = 1, split_steps = 0;   // into how many parts of how many steps K is divided (SplitK)

    uint64_t MapBytes() const { return sum == Sum::kSplit ? tiles / (uint64_t)split_parts : tiles; }   // progress bytes: one for a tile
    size_t PartialBytes() const { return sum == Sum::kSplit ? (size_t)tiles * tile * tile * 4 : 0; }
};

/// One launch, or two for rows that do not fill whole rounds of large tiles.
struct Plan
{
    Part part[2];
    int parts;
    uint64_t Tiles() const { return part[0].tiles + (parts > 1 ? part[1].tiles : 0); }
    uint64_t MapBytes() const { return part[0].MapBytes() + (parts > 1 ? part[1].tiles : 0); }
    size_t PartialBytes() const { return parts == 1 ? part[0].PartialBytes() : 0; }   // (one launch: see QuickestPlan())
};

/// A plan for copies of A, B or both with rows on 16-byte boundaries (no parts: none).
struct CopyPlan
{
    Plan plan {};
    int lda = 0, ldb = 0;                  // of what the plan's kernels read
    uint32_t a_groups = 0, b_groups = 0;   // work-groups that copy (0: the matrix stays where it is)
    size_t a_bytes = 0, b_bytes = 0;
    uint64_t Groups() const { return (uint64_t)a_groups + b_groups + plan.Tiles(); }
    size_t CopyBytes() const { return a_bytes + b_bytes; }   // (rows of whole 128-byte lines: what follows is aligned)
};

struct Plans
{
    Plan in_place;         // for A and B as they lie
    CopyPlan copies;       // for their copies
    Plan without_memory;   // as they lie, and K not divided among work-groups
    uint64_t MapBytes() const { return std::max({ in_place.MapBytes(), copies.Groups(), without_memory.MapBytes() }); }
};

class HipGemmCommand final : public HipGuardedCommand
{
public:
    HipGemmCommand(const void *A, const void *B, void *C, int M, int N, int K, const Plans &plans, int guard_mode)
        : HipGuardedCommand((uint32_t)plans.MapBytes(), guard_mode)
        , A_((const uint16_t *)A), B_((const uint16_t *)B), C_((uint16_t *)C), M_(M), N_(N), K_(K), plans_(plans) {}

protected:
    virtual void ReserveOnSubmit(HipQueue &q) override
    {
        if (decided_ || ScratchBytes() == 0) return;
        no_memory_ = q.SharedScratch()->Get(ScratchBytes()) == nullptr ||
                     (PlanWithScratch().PartialBytes() != 0 && q.SharedScratch()->Tickets() == nullptr);
    }

    /// Where copies and partial sums go is decided at the first launch: every replay takes the same way.
    virtual hipError_t PrepareLaunch(HipQueue &q) override
    {
        if (decided_ || ScratchBytes() == 0) return hipSuccess;
        decided_ = true;
        if (no_memory_) return hipSuccess;   // (as found at submission: nothing is allocated under the XQueue's locks)
        // A graph outlives the command and its queue: what is captured reads A and B themselves, and does divided K in turn.
        hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing(q.Stream(), &capture) != hipSuccess) (void)hipGetLastError();
        if (capture != hipStreamCaptureStatusNone) return hipSuccess;
        scratch_ = q.SharedScratch();
        if (PlanWithScratch().PartialBytes() != 0) {
            split_.tickets = (unsigned long long *)scratch_->Tickets();
            if (split_.tickets == nullptr) return hipSuccess;
        }
        at_ = (uint8_t *)scratch_->Get(ScratchBytes());   // nullptr: no memory, in place and in turn
        split_.partials = (float *)(at_ + plans_.copies.CopyBytes());
        return hipSuccess;
    }

    virtual hipError_t LaunchKernel(hipStream_t stream, bool guarded, const XGuardArgs &g) override
    {
        const hipEvent_t stop = TakeStopEvent();   // for the command's last kernel
        if (at_ == nullptr) return LaunchPlan(plans_.without_memory, A_, B_, K_, N_, stop, stream, guarded, g);
        // From here to the last launch no other launch that uses the buffer comes between (SharedScratch).
        std::lock_guard<std::mutex> together(scratch_->Launches());
        if (split_.tickets != nullptr) {
            split_.launch = scratch_->NextLaunch();
            if (split_.launch == 1) {
                ClearTicketsKernel<<<dim3(1), dim3(kMaxSplitTiles), 0, stream>>>(split_.tickets);
                const hipError_t err = hipGetLastError();
                if (err != hipSuccess) return err;
            }
        }
        const CopyPlan &c = plans_.copies;
        if (c.plan.parts == 0) return LaunchPlan(plans_.in_place, A_, B_, K_, N_, stop, stream, guarded, g);
        const RowCopy a { A_, (uint16_t *)at_, (uint32_t)M_, (uint32_t)K_, (uint32_t)c.lda, c.a_groups };
        const RowCopy b { B_, (uint16_t *)(at_ + c.a_bytes), (uint32_t)K_, (uint32_t)N_, (uint32_t)c.ldb, c.b_groups };
        XGuardArgs without_map = g;
        without_map.done = nullptr;
        LaunchWithStop(nullptr, guarded ? CopyRowsKernel<true> : CopyRowsKernel<false>, dim3(c.a_groups + c.b_groups), dim3(kCopyThreads), stream, a, b,
                       (const uint8_t *)(g.resume ? g.done : nullptr), (uint32_t)c.plan.MapBytes(), without_map);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        return LaunchPlan(c.plan, c.a_groups != 0 ? a.to : A_, c.b_groups != 0 ? b.to : B_, c.lda, c.ldb, stop, stream, guarded, g);
    }

private:
    /// The guard of a launch whose progress bytes follow those of a launch of `groups` work-groups.
    static XGuardArgs Behind(const XGuardArgs &g, uint64_t groups)
    {
        XGuardArgs behind = g;
        if (behind.done != nullptr) behind.done += groups;
        return behind;
    }

    hipError_t LaunchPlan(const Plan &plan, const uint16_t *A, const uint16_t *B, int lda, int ldb, hipEvent_t stop, hipStream_t stream, bool guarded, const XGuardArgs &g)
    {
        if (plan.parts == 1) return LaunchPart(plan.part[0], A, B, lda, ldb, stop, stream, guarded, g);
        const hipError_t err = LaunchPart(plan.part[0], A, B, lda, ldb, nullptr, stream, guarded, g);
        if (err != hipSuccess) return err;
        return LaunchPart(plan.part[1], A, B, lda, ldb, stop, stream, guarded, Behind(g, plan.part[0].tiles));
    }

    hipError_t LaunchPart(const Part &part, const uint16_t *A, const uint16_t *B, int lda, int ldb, hipEvent_t stop, hipStream_t stream, bool guarded, const XGuardArgs &g)
    {
        const uint16_t *const a = A + (size_t)part.first_row * lda;
        uint16_t *const c = C_ + (size_t)part.first_row * N_;
        if (part.body == Body::kAnyShape) {
            const uint32_t tiles_n = (uint32_t)((N_ + kAnyTile - 1) / kAnyTile);
            const dim3 grid((uint32_t)part.tiles), block(256);
            LaunchWithStop(stop, guarded ? GemmBf16AnyShapeKernel<true> : GemmBf16AnyShapeKernel<false>, grid, block, stream,
                           a, B, c, part.rows, N_, K_, tiles_n, g);
            return hipGetLastError();
        }
        if (part.sum != Sum::kOneGo) {
            SplitK split = split_;
            split.parts = (uint32_t)part.split_parts;
            split.steps = (uint32_t)part.split_steps;
            SplitKernel kernel = nullptr;
            switch (part.fit) {
            case Fit::kExact:     kernel = SplitKernelFor<Fit::kExact>(part, guarded); break;
            case Fit::kEdges:     kernel = SplitKernelFor<Fit::kEdges>(part, guarded); break;
            case Fit::kUnaligned: kernel = SplitKernelFor<Fit::kUnaligned>(part, guarded); break;
            }
            LaunchWithStop(stop, kernel, dim3((uint32_t)part.tiles), dim3(256), stream, a, B, c, part.rows, N_, K_, lda, ldb, g, split);
            return hipGetLastError();
        }
        Kernel kernel = nullptr;
        switch (part.fit) {
        case Fit::kExact:     kernel = KernelFor<Fit::kExact>(part, guarded); break;
        case Fit::kEdges:     kernel = KernelFor<Fit::kEdges>(part, guarded); break;
        case Fit::kUnaligned: kernel = KernelFor<Fit::kUnaligned>(part, guarded); break;   // (never large)
        }
        LaunchWithStop(stop, kernel, dim3((uint32_t)part.tiles), dim3(part.tile == kLargeTile ? 512 : 256), stream,
                       a, B, c, part.rows, N_, K_, lda, ldb, g);
        return hipGetLastError();
    }

    using Kernel = void (*)(const uint16_t *, const uint16_t *, uint16_t *, int, int, int, int, int, XGuardArgs);
    template <Fit kFit, int kTileM, int kTileN, int kWavesM, int kWavesN>
    static Kernel LargeKernelFor(bool guarded) { return guarded ? GemmBf16Kernel<true, kFit, kTileM, kTileN, kWavesM, kWavesN> : GemmBf16Kernel<false, kFit, kTileM, kTileN, kWavesM, kWavesN>; }
    template <Fit kFit>
    static Kernel KernelFor(const Part &part, bool guarded)
    {
        if constexpr (kFit == Fit::kExact) {
            if (part.body == Body::kTwoBuffers && part.tile == kSmallTile) return LargeKernelFor<kFit, kSmallTile, kSmallTile, 2, 2>(guarded);
        }
        if constexpr (kFit != Fit::kUnaligned) {
            if (part.tile == kLargeTile && part.tile_rows == kThreeQuarterRows) return LargeKernelFor<kFit, kThreeQuarterRows, kLargeTile, 2, 4>(guarded);
            if (part.tile == kLargeTile && part.tile_rows == kHalfRows) return LargeKernelFor<kFit, kHalfRows, kLargeTile, 2, 4>(guarded);
            if (part.tile == kLargeTile) return LargeKernelFor<kFit, kLargeTile, kLargeTile, 2, 4>(guarded);
        }
        if (part.tile == kSmallTile) return guarded ? GemmDeepKernel<true, kFit, kSmallTile, 4> : GemmDeepKernel<false, kFit, kSmallTile, 4>;
        return guarded ? GemmDeepKernel<true, kFit, kTinyTile, 4> : GemmDeepKernel<false, kFit, kTinyTile, 4>;
    }

    using SplitKernel = void (*)(const uint16_t *, const uint16_t *, uint16_t *, int, int, int, int, int, XGuardArgs, SplitK);
    template <Fit kFit>
    static SplitKernel SplitKernelFor(const Part &part, bool guarded)
    {
        return part.sum == Sum::kSplit ? SplitKernelFor<kFit, Sum::kSplit>(part, guarded) : SplitKernelFor<kFit, Sum::kInTurn>(part, guarded);
    }
    template <Fit kFit, Sum kSum>
    static SplitKernel SplitKernelFor(const Part &part, bool guarded)
    {
        if (part.tile == kSmallTile) return guarded ? GemmSplitKernel<true, kFit, kSmallTile, 4, kSum> : GemmSplitKernel<false, kFit, kSmallTile, 4, kSum>;
        return guarded ? GemmSplitKernel<true, kFit, kTinyTile, 4, kSum> : GemmSplitKernel<false, kFit, kTinyTile, 4, kSum>;
    }

    /// The plan where there is memory for copies and partial sums, and how much that takes.
    const Plan &PlanWithScratch() const { return plans_.copies.plan.parts != 0 ? plans_.copies.plan : plans_.in_place; }
    size_t ScratchBytes() const { return plans_.copies.CopyBytes() + PlanWithScratch().PartialBytes(); }

    const uint16_t *A_, *B_;
    uint16_t *C_;
    const int M_, N_, K_;
    const Plans plans_;
    std::shared_ptr<class SharedScratch> scratch_;
    uint8_t *at_ = nullptr;   // the copies, A's first, then partial sums; nullptr: plans_.without_memory
    SplitK split_ {};
    bool decided_ = false, no_memory_ = false;
};

inline uint64_t TilesOf(int M, int N, int tile_rows, int tile)
{
    return ((uint64_t)M + (unsigned)tile_rows - 1) / (unsigned)tile_rows * (((uint64_t)N + (unsigned)tile - 1) / (unsigned)tile);
}
inline uint64_t TilesOf(int M, int N, int tile) { return TilesOf(M, N, tile, tile); }

inline uint32_t ComputeUnits()
{
    static const uint32_t cus = []() {
        int dev = 0, n = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        return (uint32_t)(n > 0 ? n : 256);
    }();
    return cus;
}

/// Whether the rows of a matrix of `cols` columns start on 16-byte boundaries.
inline bool Aligned(const void *matrix, int cols) { return ((uintptr_t)matrix & 15) == 0 && cols % 8 == 0; }
inline bool Aligned(const void *A, const void *B, const void *C, int N, int K) { return Aligned(A, K) && Aligned(B, N) && Aligned(C, N); }

/// XSCHED_HIP_GEMM_TILE: 64, 128 or 256, else 0.
inline int ForcedTile()
{
    int64_t forced = 0;
    GetEnvInt64("XSCHED_HIP_GEMM_TILE", forced);
    return forced == kTinyTile || forced == kSmallTile || forced == kLargeTile ? (int)forced : 0;
}

/// XSCHED_HIP_GEMM_TILE_ROWS beside XSCHED_HIP_GEMM_TILE=256: 128, 192 or 256 (the default).
inline int ForcedTileRows()
{
    int64_t rows = 0;
    GetEnvInt64("XSCHED_HIP_GEMM_TILE_ROWS", rows);
    return rows == kHalfRows || rows == kThreeQuarterRows ? (int)rows : kLargeTile;
}

/// What a plan may assume: rows of A and B (or of their copies), and rows of C, start on 16-byte boundaries.
struct Rows { bool inputs, output; };

inline Part PartOf(int first_row, int rows, int N, int K, Rows aligned, int tile, int tile_rows)
{
    const bool exact = aligned.inputs && aligned.output && rows % tile_rows == 0 && N % tile == 0 && K % kStepK == 0;
    return Part { first_row, rows, tile, exact ? Fit::kExact : aligned.inputs ? Fit::kEdges : Fit::kUnaligned,
                  tile == kLargeTile ? Body::kTwoBuffers : Body::kFourStages, TilesOf(rows, N, tile_rows, tile), tile_rows };
}
inline Part PartOf(int first_row, int rows, int N, int K, Rows aligned, int tile) { return PartOf(first_row, rows, N, K, aligned, tile, tile); }

/// Roughly how long a part takes, in us: a launch, then rounds of one tile per compute unit (two of
/// 128 x 128 with two buffers), each with its first loads and its write-out, the last round quicker the fewer
/// units it keeps busy: in proportion, or, on tiles of 192 x 256, only where few units idle (the cube: a full round runs
/// against the power limit, and units that idle leave the others a higher clock; the rates of 256 x 256 are fitted without
/// it, for their choice between one launch and two: with it 4992^3 is slower by 3 %). The rates are fitted to outputs of 4 to 4096 tiles of 128 x 128 at
/// K from 128 to 8192. Of 150 products drawn from 128 to 8192 in each dimension, half of them ragged, each timed on every tile, what the
/// plan takes is 1.2 % behind the quickest on average; 14 % at most where K is not divided (272 x 7184 x 288 7.9 us, 7.0 on
/// tiles of 128) and 28 % where it is (561 x 456 x 2312 13.6, 10.6 in more parts).
inline double MicrosOf(const Part &part, int K, double pace = 1.0 /* of the steps */)
{
    // us of a round, and per K step of a full round and of one with a single tile: [exact, edges, unaligned]
    struct Rates { double round, full, single; };
    constexpr Rates large[3] = { { 5.0, 1.36, 1.00 }, { 5.0, 1.43, 1.05 }, {} };
    constexpr Rates three_quarters[3] = { { 4.5, 1.08, 0.80 }, { 5.0, 1.17, 0.86 }, {} };
    constexpr Rates half[3] = { { 3.5, 0.82, 0.66 }, { 3.5, 0.86, 0.66 }, {} };
    constexpr Rates pair = { 1.7, 0.90, 0.45 };
    constexpr Rates small[3] = { { 2.5, 0.45, 0.37 }, { 2.5, 0.53, 0.41 }, { 2.5, 0.69, 0.48 } };
    constexpr Rates tiny[3] = { { 0.5, 0.195, 0.14 }, { 0.5, 0.25, 0.16 }, { 0.5, 0.32, 0.29 } };
    const bool two_per_unit = part.tile == kSmallTile && part.body == Body::kTwoBuffers;
    const bool power_bound = part.tile == kLargeTile && part.tile_rows == kThreeQuarterRows;
    const Rates *const of_large = part.tile_rows == kLargeTile ? large : part.tile_rows == kThreeQuarterRows ? three_quarters : half;
    const Rates &r = two_per_unit ? pair : (part.tile == kLargeTile ? of_large : part.tile == kSmallTile ? small : tiny)[(int)part.fit];
    const double rounds = (double)part.tiles / ((two_per_unit ? 2 : 1) * ComputeUnits()), whole = std::floor(rounds);
    const double busy = power_bound ? (rounds - whole) * (rounds - whole) * (rounds - whole) : rounds - whole;
    const double step = whole * r.full + (rounds > whole ? r.single + (r.full - r.single) * busy : 0.0);
    return 3.0 + std::ceil(rounds) * r.round + pace * step * ((K + kStepK - 1) / kStepK);
}

inline double MicrosOf(const Plan &plan, int K, double pace = 1.0)
{
    double us = 0.0;
    for (int i = 0; i < plan.parts; ++i) us += MicrosOf(plan.part[i], K, pace);
    return us;
}

/// Whether K is so short that the any-shape kernel is the quickest: up to 32, one step of it;
/// further for outputs of many tiles, whose write-out it overlaps best, and the further the fewer of
/// its loads come one by one. Measured on either side, any-shape kernel against the quickest of the others, us:
/// with 16-byte rows in all three matrices, 7000^2 at K = 64 35.9 against 41.6, at 72 47.5 against
/// 47.6, 4000 x 4008 at 64 14.8 against 13.7; with 16-byte rows in A, 7001 x 7003 at 128 84 against 102, at 160 103 against
/// 96, 8191 x 515 at 96 12.1 against 13.9, at 128 14.4 against 13.9, 2000 x 1999 at 64 9.0 against
/// 9.4, at 72 10.5 against 10.3, 1000 x 1001 at 40 5.5 against 5.3; without, 2000 x 1999 at 31 8.3 against 9.4, at 33
/// 9.5 against 9.9, at 63 13.3 against 9.5, 4001 x 4003 at 31 18.6 against 31.2, at 63 36.8 against 31.4.
/// Where rows of C are whole 64-byte pieces the other kernels write them as fast as memory takes them, and
/// what the any-shape kernel can win is a last round of large tiles that is at most half full. Passes, us:
/// 4096^2 at 32 (one whole round) 25.6 against 20.0, 8192^2 at 32 (four) 56.5 against 49.3, 6353 x 7168 at 32 (2.7)
/// 43.7 against 38.1, at 64 47.0 against 41.1; 4400 x 4096 at 32 (1.1) 26.2 against 27.9, 6400 x 8192 (3.1) 42.6
/// against 45.7, 7912 x 4800 (2.3) 35.3 against 38.4, but at 64 41.3 against 39.0. (With rows of other lengths,
/// 6353 x 7176 at 64: 49.4 against 57.5.)
inline bool ShortK(const void *A, const void *B, const void *C, int M, int N, int K)
{
    const uint64_t tiles = TilesOf(M, N, kAnyTile), units = ComputeUnits();
    if (tiles > GuardState::kMaxWorkGroups) return false;
    int limit = 32;
    if (Aligned(A, B, C, N, K)) {
        if (N % 32 == 0) {
            const uint64_t large = TilesOf(M, N, kLargeTile), over = large % units;
            if (large < units || over == 0 || 2 * over > units) limit = 0;
        } else if (tiles >= 32 * units) {
            limit = 64;
        }
    } else if (((uintptr_t)A & 15) == 0 && K % 8 == 0) {
        limit = tiles >= 12 * units ? 128 : 2 * tiles >= 9 * units ? 96 : tiles >= 4 * units ? 64 : 32;
    } else if (tiles > 4 * units) {
        limit = 48;
    }
    return K <= limit;
}

constexpr int kLeastSplitSteps = 17;   // below, less than a us can be won
constexpr int kLeastPartSteps = 8;
/// What a split adds: the partial sums on their way past the L2, the ticket, and the last group's way
/// through all parts. Fitted to the products of QuickestPlan()'s comment, and a us more: what is won in a stream
/// of commands is partly lost again where a command is waited for alone.
inline double SplitMicros(const Part &part)
{
    const double parts = part.split_parts, groups = (double)part.tiles;
    return part.tile == kSmallTile ? 1.0 + 0.3 * parts + 0.015 * groups : 0.5 + 0.25 * parts + 0.012 * groups;
}

inline double MicrosOfPlan(const Plan &plan, int K, double pace = 1.0)
{
    const Part &first = plan.part[0];
    return first.sum == Sum::kSplit ? MicrosOf(first, first.split_steps * kStepK, pace) + SplitMicros(first) : MicrosOf(plan, K, pace);
}

/// All of C with K divided into parts of split_steps steps.
inline Part SplitPartOf(int M, int N, int K, Rows aligned, int tile, int split_steps)
{
    Part part = PartOf(0, M, N, K, aligned, tile);
    part.sum = Sum::kSplit;
    part.split_steps = split_steps;
    part.split_parts = ((K + kStepK - 1) / kStepK + split_steps - 1) / split_steps;
    part.tiles *= (uint64_t)part.split_parts;
    return part;
}

/// Whether the work-groups of a split part have a compute unit each.
inline bool CanSplit(const Part &part) { return part.MapBytes() <= kMaxSplitTiles && part.tiles <= ComputeUnits(); }

/// The plan for a shape: the quickest by the estimate above of one launch on large, small or tiny
/// tiles and of two, large tiles for the rows that fill whole tiles, or whole rounds of them, and
/// whatever is quickest for the rest. Large tiles have 256 columns and 256, 192 or 128 rows: outputs of 150 to 250 tiles of 256 x 256 leave
/// compute units idle that 192 rows keep busy, ragged ones of 257 to 512 tiles of 128 x 128 are one round of 128 x 256 (us per command, without
/// these and with them: 3072^3 57.4 -> 49.8, 3456 x 3456 x 512 18.0 -> 15.2, 7451 x 2632 x 1232 69.2 -> 56.8, 5801 x 760 x 3344 59.4 -> 51.3, 805 x 7704 x 104 12.1 -> 9.6). Large tiles do more arithmetic per byte read from LDS, but a
/// round of few tiles leaves compute units idle (pass times in us, large and small tiles as they were
/// chosen before by the share of the compute units covered and by exact multiples only, and now:
/// 8197 x 8192 x 8192 1038 -> 836, 4100 x 4096 x 4096 156 -> 130, 6016 x 6016 x 8192 564 -> 485,
/// 6000 x 6008 x 6000 539 -> 424, 4000^3 146 -> 114; 4096^3 106 per command on large tiles against
/// 126 on small ones, 2048^3 20.9 on small against 30.1 on tiny ones, 1024^3 5.8 on tiny ones against
/// 9.4 on small ones). Rows without 16-byte alignment do not go straight into LDS, which the large
/// tiles need (a tile on its way through registers beside their accumulators does not fit).
/// Where tiny or small tiles leave compute units idle and K is long, K is divided (SplitK). us per command, whole / in 2 / 3 / 4 /
/// 8 / 16 parts on tiles of 64: 128 x 128 x 8192 22.7 / 14.1 / 11.3 / 10.3 / 9.8 / 10.5, 256 x 256 x 4096 13.6 / 9.3 / 9.1 /
/// 9.5 / 10.0 / 12.5, x 2048 8.5 / 8.1 / 8.2 / 8.7 / 9.5, 512 x 512 x 2048 9.0 / 8.5 / 9.1 / 10.1, 500 x 499 x 4095
/// 23.4 / 15.4 / 13.2 / 13.5; whole on tiles of 64 / in 2 / 3 / 4 parts on tiles of 128: 1024 x 1024 x 8192 31.5 / 28.9 /
/// 26.0 / 27.7, 1000 x 999 x 8001 44.3 / 46.6 / 36.9 / 34.4, but 1024 x 1024 x 4096 17.5 / 18.5 / 18.6 / 20.5.
/// How is decided once for a shape (SplitStepsFor()); here parts of split_steps steps are given, 0: K in one go.
/// XSCHED_HIP_GEMM_TILE=64|128|256 overrides the tile where the shape allows (128: four stages), and K is not divided.
/// A plan of more tiles than the progress map holds is passed over for one that fits: 13413745 x
/// 1280 x 1024, 262025 tiles by the count below, would be quickest as two launches of 262295.
inline Plan QuickestPlan(int M, int N, int K, Rows aligned, int split_steps)
{
    if (split_steps != 0) {
        Plan best {};
        for (const int tile : { kTinyTile, kSmallTile }) {
            const Plan split { { SplitPartOf(M, N, K, aligned, tile, split_steps), {} }, 1 };
            if (CanSplit(split.part[0]) && (best.parts == 0 || MicrosOfPlan(split, K) < MicrosOfPlan(best, K))) best = split;
        }
        return best;
    }
    auto best_part = [&](int first_row, int rows) {
        Part best = PartOf(first_row, rows, N, K, aligned, kSmallTile);
        if (best.fit == Fit::kExact) {
            Part two_per_unit = best;
            two_per_unit.body = Body::kTwoBuffers;
            if (MicrosOf(two_per_unit, K) < MicrosOf(best, K)) best = two_per_unit;
        }
        for (const int tile : { kTinyTile, kLargeTile }) {
            if (tile == kLargeTile && !aligned.inputs) continue;
            const Part other = PartOf(first_row, rows, N, K, aligned, tile);
            const bool fits = other.tiles <= GuardState::kMaxWorkGroups, best_fits = best.tiles <= GuardState::kMaxWorkGroups;
            if (fits && (!best_fits || MicrosOf(other, K) < MicrosOf(best, K))) best = other;
        }
        return best;
    };
    Plan best { { best_part(0, M), {} }, 1 };
    double least = MicrosOf(best.part[0], K);
    auto consider = [&](int64_t large_rows) {
        if (!aligned.inputs || large_rows <= 0 || large_rows >= M) return;
        const Part first = PartOf(0, (int)large_rows, N, K, aligned, kLargeTile), rest = best_part((int)large_rows, M - (int)large_rows);
        const double both = MicrosOf(first, K) + MicrosOf(rest, K);
        if (first.tiles + rest.tiles > GuardState::kMaxWorkGroups) return;
        if (both < least) { least = both; best = Plan { { first, rest }, 2 }; }
    };
    consider((int64_t)(M / kLargeTile) * kLargeTile);                       // all whole large tiles
    const int64_t in_row = (N + kLargeTile - 1) / kLargeTile;                // all whole rounds of large tiles
    const int64_t whole_rounds = (int64_t)TilesOf(M, N, kLargeTile) / ComputeUnits();
    consider(whole_rounds * ComputeUnits() / in_row * kLargeTile);
    // All of C on large tiles of fewer rows. Of 140 products that are quickest in two launches otherwise, half of them ragged, 40 are quicker on these by
    // the estimate: they take 0.94 of the time on average, 1.03 at most (3072 x 7808 x 7488 290.2 -> 297.8 us; 4608^3 161.6 -> 154.1, 4994 x 6840 x 456
    // 58.7 -> 55.1, 3488 x 5808 x 464 36.9 -> 32.3, 2624 x 7296 x 6400 245 -> 221). Asking them to be quicker by a tenth left 31 of the 40 in two launches.
    if (aligned.inputs) {
        for (const int tile_rows : { kThreeQuarterRows, kHalfRows }) {
            const Part part = PartOf(0, M, N, K, aligned, kLargeTile, tile_rows);
            if (part.tiles > GuardState::kMaxWorkGroups) continue;
            const double us = MicrosOf(part, K);
            if (us < least) { least = us; best = Plan { { part, {} }, 1 }; }
        }
    }
    return best;
}

constexpr size_t kMaxScratchBytes = SharedScratch::kMaxBytes;   // copies of A and B and partial sums together
// What copies cost by the estimate, fitted to 21 products of 300 x 301 x 6001 to 4000 x 3999 x 301, each timed in place and on
// copies. It errs towards in place: of those in PlansFor()'s comment 2000 x 1999 x 3001 and 3000 x 2999 x 301 and x 101 stay there
// though copies are quicker.
constexpr double kCopyMicros = 8.0;                 // launch of the copying kernel and the one behind it,
constexpr double kCopyRate = 12e6;                  // bytes per us, read and written, as long as matrices and copies stay in the last-level
constexpr double kCachedCopyBytes = 100e6;          // cache (256 MB): up to so many bytes of copies,
constexpr double kFarCopyRate = 3.5e6;              // and for those beyond, with reading them again from memory,
constexpr double kCopyPace = 0.85;                  // time of a step on rows of whole cache lines against any rows on 16-byte boundaries

inline double CopyMicros(const CopyPlan &p)
{
    const double cached = std::min((double)p.CopyBytes(), kCachedCopyBytes);
    return kCopyMicros + 2.0 * cached / kCopyRate + 2.0 * ((double)p.CopyBytes() - cached) / kFarCopyRate;
}

/// What the estimate misses of copies that are multiplied on large tiles of fewer rows, in us: behind a short K they lose to
/// in place by what was copied of B, and a little of what was of A. Of 156 products that the estimate alone takes from in place to
/// such tiles, all timed both ways and none with more than kCachedCopyBytes of copies (for those kFarCopyRate is fitted with them), 105 stay on them with this: 0.907 of the time in place on average (1205 x 5002 x 1440 32.2 us in place,
/// 34.6 on copies at worst; 767 x 5952 x 1317 31.8 and 25.8, 1750 x 4884 x 336 22.8 and 19.4), and 51 go back: copies took 1.017 of their
/// time in a stream of commands and 1.046 of a pass (897 x 4134 x 1120 24.5 and 29.6, 1897 x 3814 x 1002 27.2 and 30.3,
/// 774 x 6505 x 1056 30.8 and 33.9; but 671 x 6179 x 1661 44.2 and 39.5). Of more than 30 MB of B or 60 of A no more than for
/// those: 640 x 12001 x 3801 (91 MB of B) 114.4 in place and 98.9, 730 x 7489 x 2278 (35 MB) 57.8 and 53.0, but 400 x 8191 x 4001 (66 MB) 56.3 and 62.6.
/// Of 30000 drawn products of up to 16384 x 16384 x 8192 that went on copies to other tiles one changes its way by it (11157 x 633 x 2629 65.3 in place and 69.6).
inline double FewerRowsMicros(const CopyPlan &p, int K)
{
    const Part &part = p.plan.part[0];
    return part.tile_rows == part.tile || K <= 7 * kStepK || (double)p.CopyBytes() > kCachedCopyBytes ? 0.0 : 0.23e-6 * std::min((double)p.b_bytes, 30e6) + 0.04e-6 * std::min((double)p.a_bytes, 60e6);
}

/// Copies of A, B or both without a plan for them; without copies where they are too large.
inline CopyPlan CopiesFor(bool copy_a, bool copy_b, int M, int N, int K)
{
    CopyPlan p;
    p.lda = copy_a ? (K + 63) / 64 * 64 : K;
    p.ldb = copy_b ? (N + 63) / 64 * 64 : N;
    p.a_bytes = copy_a ? (size_t)M * p.lda * 2 : 0;
    p.b_bytes = copy_b ? (size_t)K * p.ldb * 2 : 0;
    if (p.CopyBytes() > kMaxScratchBytes || K > kMaxK - 64 || N > kMaxK - 64) return CopyPlan {};
    p.a_groups = copy_a ? CopyGroups(M, p.lda) : 0;
    p.b_groups = copy_b ? CopyGroups(K, p.ldb) : 0;
    return p;
}

/// Steps of the parts that K is divided into, 0: it is not. Of all ways on tiles of 64 and 128 the one that the quickest plan
/// takes for rows on 16-byte boundaries wherever N and K allow that, with memory: every other plan for the same
/// sizes divides K alike, so that a product's bits don't depend on where its matrices lie, on capture or on memory.
/// (What it costs: an element behind a 16-byte boundary 640 x 640 x 3072 takes 24.4 us, 16.5 in the two parts that are best there; 1024 x
/// 1024 x 4096 31.6 and 29.4.) Parts of an even number of steps, for add_ended_part().
inline int SplitStepsFor(int M, int N, int K)
{
    const int steps = (K + kStepK - 1) / kStepK;
    if (steps < kLeastSplitSteps || 2 * TilesOf(M, N, kSmallTile) > ComputeUnits()) return 0;
    int best = 0;
    double least = 0.0;
    bool first = true;
    auto consider = [&](Rows rows, double copying, double pace) {
        const double whole = copying + MicrosOf(QuickestPlan(M, N, K, rows, 0), K, pace);
        if (first || whole < least) { least = whole; best = 0; }
        first = false;
        for (const int tile : { kTinyTile, kSmallTile }) {
            for (int parts = 2; ; ++parts) {
                const int split_steps = ((steps + parts - 1) / parts + 1) / 2 * 2;
                const Plan split { { SplitPartOf(M, N, K, rows, tile, split_steps), {} }, 1 };
                if (split_steps < kLeastPartSteps || !CanSplit(split.part[0])) break;
                if (steps - (split.part[0].split_parts - 1) * split_steps < kLeastLastSteps) continue;
                const double us = copying + MicrosOfPlan(split, K, pace);
                if (us < least) { least = us; best = split_steps; }
            }
        }
    };
    const Rows rows { K % 8 == 0 && N % 8 == 0, N % 8 == 0 };
    consider(rows, 0.0, 1.0);
    if (!rows.inputs) {
        const CopyPlan copies = CopiesFor(K % 8 != 0, N % 8 != 0, M, N, K);
        if (copies.CopyBytes() != 0) consider(Rows { true, rows.output }, CopyMicros(copies), kCopyPace);
    }
    return best;
}

/// How a product is computed: with the matrices as they lie, on copies of whichever of A and B has rows off 16-byte
/// boundaries (if that is quicker), and without memory. Through registers a step waits for loads at any multiple of two
/// bytes, each 128-byte piece of a row in two cache lines (0.7 us against 0.45 for 128 x 128 tiles of 64 k), and large tiles do not fit; the copies cost
/// their launch and two passes over the matrices (8191^2 elements 87 us = 6.2 TB/s with what is
/// written, 2000 x 2047 and 2047 x 1999 together 9.5). Rows of the copies are whole 128-byte lines (rows of 2000 and
/// 2048 elements rather than of 2048: 27 us for the 2000 x 1999 x 2047 that takes 23.5). us per command,
/// in place / on copies: 500 x 499 x 4095 13.5 / 17.9; 1500 x 1499 x 4095 44.2 / 39.6, x 2047 25.8 / 28.1; 2000 x 1999
/// x 2047 31.0 / 31.2, x 3001 43.3 / 38.1, x 4095 56.3 / 46.5; 2500 x 2501 x 1001 32.5 / 32.1; 3000 x 2999 x 301
/// 27.9 / 22.7, x 101 24.3 / 18.5; 4000 x 3999 x 301 38.4 / 30.1; 1000 x 999 x 8001 36.8 / 39.9; 128 x 8191 x 8191
/// 48.9 / 82.0. Above the size of the last-level cache (copies on large tiles of any rows): 8191 x 511 x 8191 89.5 / 113, 500 x 12287 x 8191 166 / 211, 16383 x 300 x
/// 8191 162 / 239, 512 x 16383 x 8191 216 / 247, but 8191 x 767 x 8191 165 / 151, 700 x 8191 x 8191 176 / 151, 8191 x 1023 x 8191 180 / 164, 600 x 16383 x 4095
/// 138 / 126, 900 x 16383 x 4095 204 / 148, 8191 x 2047 x 8191 359 / 254. A pass of 8191^3 1791 / 918.
inline Plans PlansFor(const void *A, const void *B, const void *C, int M, int N, int K, int forced)
{
    Plans plans {};
    plans.in_place = Plan { { Part { 0, M, kAnyTile, Fit::kUnaligned, Body::kAnyShape, TilesOf(M, N, kAnyTile), kAnyTile }, {} }, 1 };
    plans.without_memory = plans.in_place;
    if (N < 8 || (int64_t)M * K < 8 || K > kMaxK || N > kMaxK) return plans;
    if (forced == 0 && ShortK(A, B, C, M, N, K)) return plans;
    const bool a_aligned = Aligned(A, K), b_aligned = Aligned(B, N);
    const Rows aligned { a_aligned && b_aligned, Aligned(C, N) };
    if (forced != 0 && (forced != kLargeTile || aligned.inputs)) {
        plans.in_place = Plan { { PartOf(0, M, N, K, aligned, forced, forced == kLargeTile ? ForcedTileRows() : forced), {} }, 1 };
        plans.without_memory = plans.in_place;
        return plans;
    }
    const int split_steps = forced == 0 ? SplitStepsFor(M, N, K) : 0;
    plans.in_place = QuickestPlan(M, N, K, aligned, split_steps);
    plans.without_memory = plans.in_place;
    if (split_steps != 0) {
        Part &part = plans.without_memory.part[0];
        const int parts = part.split_parts;
        part = PartOf(0, M, N, K, aligned, kTinyTile);
        if (const Part small = PartOf(0, M, N, K, aligned, kSmallTile); MicrosOf(small, K) < MicrosOf(part, K)) part = small;
        part.sum = Sum::kInTurn;
        part.split_parts = parts;
        part.split_steps = split_steps;
    }
    if (forced != 0 || aligned.inputs) return plans;
    CopyPlan copies = CopiesFor(!a_aligned, !b_aligned, M, N, K);
    if (copies.CopyBytes() == 0) return plans;
    copies.plan = QuickestPlan(M, N, K, Rows { true, aligned.output }, split_steps);
    if (copies.Groups() > GuardState::kMaxWorkGroups || copies.CopyBytes() + copies.plan.PartialBytes() > kMaxScratchBytes) return plans;
    if (CopyMicros(copies) + FewerRowsMicros(copies, K) + MicrosOfPlan(copies.plan, K, kCopyPace) < MicrosOfPlan(plans.in_place, K)) plans.copies = copies;
    return plans;
}

/// Tiles by which a shape is accepted or refused. They are the tiles of the kernels that such shapes
/// once ran on: 128 x 128 or 256 x 256 for the rows up to the last multiple of 128 where everything
/// else is a multiple of the tiles, and 64 x 64.
inline uint64_t CountedTiles(const void *A, const void *B, const void *C, int M, int N, int K, int forced)
{
    const int whole = M / kSmallTile * kSmallTile;
    if (forced == kTinyTile || whole == 0 || !Aligned(A, B, C, N, K) || N % kSmallTile != 0 || K % kStepK != 0 || K > kMaxK || N > kMaxK) {
        return TilesOf(M, N, kAnyTile);
    }
    const int tile = whole % kLargeTile == 0 && N % kLargeTile == 0 && forced != kSmallTile ? kLargeTile : kSmallTile;
    return TilesOf(whole, N, tile) + TilesOf(M - whole, N, kAnyTile);
}

} // namespace gemm

} // namespace xsched::hip

using namespace xsched::hip;

static void PutParts(const gemm::Plan &plan, int32_t *out)
{
    for (int i = 0; i < 8; ++i) out[i] = 0;
    for (int i = 0; i < plan.parts; ++i) {
        const gemm::Part &part = plan.part[i];
        out[4 * i + 0] = part.rows;
        out[4 * i + 1] = part.tile;
        out[4 * i + 2] = (int32_t)part.body;
        out[4 * i + 3] = (int32_t)part.fit;
    }
}

EXPORT_C_FUNC XResult HipGemmBf16PlanOf(const void *A, const void *B, const void *C, int M, int N, int K, int32_t *out)
{
    if (out == nullptr || M <= 0 || N <= 0 || K <= 0) return kXSchedErrorInvalidValue;
    PutParts(gemm::PlansFor(A, B, C, M, N, K, gemm::ForcedTile()).in_place, out);
    return kXSchedSuccess;
}

EXPORT_C_FUNC XResult HipGemmBf16CopyPlanOf(const void *A, const void *B, const void *C, int M, int N, int K, int32_t *out)
{
    if (out == nullptr || M <= 0 || N <= 0 || K <= 0) return kXSchedErrorInvalidValue;
    const gemm::CopyPlan copies = gemm::PlansFor(A, B, C, M, N, K, gemm::ForcedTile()).copies;
    PutParts(copies.plan, out);
    out[8] = (int32_t)copies.a_groups;
    out[9] = (int32_t)copies.b_groups;
    return kXSchedSuccess;
}

EXPORT_C_FUNC XResult HipGemmBf16TileRowsOf(const void *A, const void *B, const void *C, int M, int N, int K, int32_t *out)
{
    if (out == nullptr || M <= 0 || N <= 0 || K <= 0) return kXSchedErrorInvalidValue;
    const gemm::Plans plans = gemm::PlansFor(A, B, C, M, N, K, gemm::ForcedTile());
    for (int i = 0; i < 2; ++i) {
        out[i] = i < plans.in_place.parts ? plans.in_place.part[i].tile_rows : 0;
        out[2 + i] = i < plans.copies.plan.parts ? plans.copies.plan.part[i].tile_rows : 0;
    }
    return kXSchedSuccess;
}

EXPORT_C_FUNC XResult HipGemmBf16SplitsOf(const void *A, const void *B, const void *C, int M, int N, int K, int32_t *out)
{
    if (out == nullptr || M <= 0 || N <= 0 || K <= 0) return kXSchedErrorInvalidValue;
    const gemm::Plans plans = gemm::PlansFor(A, B, C, M, N, K, gemm::ForcedTile());
    out[0] = plans.in_place.part[0].split_parts;
    out[1] = plans.copies.plan.parts != 0 ? plans.copies.plan.part[0].split_parts : 0;
    return kXSchedSuccess;
}

EXPORT_C_FUNC XResult HipGemmBf16TicketsOf(HwQueueHandle hwq, uint64_t *out)
{
    if (out == nullptr) return kXSchedErrorInvalidValue;
    auto q = std::dynamic_pointer_cast<HipQueue>(HwQueueManager::Get(hwq));
    if (q == nullptr) return kXSchedErrorNotFound;
    SharedScratch &scratch = *q->SharedScratch();
    std::lock_guard<std::mutex> together(scratch.Launches());
    for (uint32_t i = 0; i < SharedScratch::kTicketWords; ++i) out[i] = 0;
    out[SharedScratch::kTicketWords] = scratch.LastLaunch();
    if (scratch.LastLaunch() == 0) return kXSchedSuccess;
    return hipMemcpy(out, scratch.Tickets(), SharedScratch::kTicketWords * sizeof(uint64_t), hipMemcpyDeviceToHost) == hipSuccess ? kXSchedSuccess : kXSchedErrorHardware;
}

EXPORT_C_FUNC XResult HipGemmBf16CommandCreate(HwCommandHandle *cmd, const void *A, const void *B,
                                               void *C, int M, int N, int K, int guard)
{
    if (cmd == nullptr || A == nullptr || B == nullptr || C == nullptr || guard < 0 || guard > 3) {
        return kXSchedErrorInvalidValue;
    }
    if (M <= 0 || N <= 0 || K <= 0 || (((uintptr_t)A | (uintptr_t)B | (uintptr_t)C) & 1) != 0) {
        XWARN("HipGemmBf16CommandCreate: M, N and K must be positive and the matrices aligned to their elements (got %d %d %d)", M, N, K);
        return kXSchedErrorInvalidValue;
    }
    const int forced = gemm::ForcedTile();
    const gemm::Plans plans = gemm::PlansFor(A, B, C, M, N, K, forced);
    // one progress-map byte per tile
    if (plans.in_place.Tiles() > GuardState::kMaxWorkGroups || gemm::CountedTiles(A, B, C, M, N, K, forced) > GuardState::kMaxWorkGroups) {
        XWARN("HipGemmBf16CommandCreate: %d x %d needs more than 2^18 tiles", M, N);
        return kXSchedErrorInvalidValue;
    }
    *cmd = HwCommandManager::Add(std::make_shared<gemm::HipGemmCommand>(A, B, C, M, N, K, plans, guard));
    return kXSchedSuccess;
}
