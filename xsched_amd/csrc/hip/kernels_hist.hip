// Guarded integer histogram for gfx950: bins[keys[i]] += 1, keys int32 in
// [0, n_bins), n_bins <= 65536, bins uint32.
//
// The keys are read once (4 bytes per key). Two things used to cost more than that read
// on MI355X: the LDS atomics when many lanes of a wave add to ONE address (the hottest bins of
// a skewed distribution; spread over addresses they are cheap: with 16 waves issuing, a CU
// retires a 64-lane ds_add every 1.7 ns on per-lane words and every 2.2 ns on random words,
// five times what this kernel asks of it) and the merge of the
// per-group counts into the one result array (device-wide atomic adds retire at
// ~90-110 G/s however they are arranged, and 256 groups times 65536 bins is a lot of
// them; hence the second kernel below).
//
// One work-group of 1024 threads owns a contiguous chunk of keys
// (sized so that a launch has about one work-group per CU) and keeps everything it
// counts on chip until the end, in 80 KiB of LDS counters split in two. Bins below 255 (two
// thirds of all Zipf(1.1) keys, a fifth of them in bins 0 and 1) have sixteen 32-bit counters
// each, one per lane modulo 16, so that at most four lanes of a wave add to the same address, no
// vote and no popcount is needed, and they cannot overflow (64, one per lane, where n_bins leaves
// the room, and then for bin 255 too, which is all that 256 bins have: 2^26 evenly spread keys over 1000 bins,
// a quarter of them in these bins, 54.7 us a pass through a queue against 56.8 with 16). Half of a compute unit's LDS and of its wave slots: two groups of different
// queues share it, and one streams keys while the other clears, writes out or waits for its first
// keys (four queues of 2^26 keys each 217 -> 207 us; with 64 counters for every one of these bins
// and 128 KiB, a group had its unit to itself). Every other bin shares one of 16384
// words with the bins 16384, 32768 and 49152 above it, as far as there are such bins: a BYTE
// each when n_bins > 32768, a half word each when n_bins > 16384, the whole word otherwise; one
// ds_add of 1 << (width * (key >> 14)) per key. One vote per iteration tells whether every key
// of the wave is below n_bins, so the add needs no branch.
//
// A byte overflows only when one bin outside the first 255 takes 256 keys of a chunk (0.1 % of
// it; the hottest such bin of a Zipf(1.1) chunk takes 80), a half when it takes 65536. Every
// overflow lowers the sum of all counters by at least 255 and nothing raises it, so "sum of
// counters == keys that must be in them" (all key slots of the chunk minus the invalid ones)
// proves there was none; a group that fails the test recounts its chunk the slow way (32-bit
// counters, a pass over its keys for every 16384 bins, atomic sweep into the result). Runs of one key
// (sorted or constant keys) in long chunks are added a thread's four keys at a time, and the recount of
// a group that saw some passes over the quarters of the bins that have no keys: 2^26 equal keys outside the
// first 255 of 65536 bins 559 -> 130 us, 2^22 78 -> 27, sorted 2^22 over 20000 bins 34.5 -> 18.3. Whole words need no test:
// with bytes for any n_bins, 2^26 evenly spread keys over 1000 bins overflowed in every group
// (262 keys of a chunk to a bin): 186 us a launch, 42 with whole words (a pass through a queue 199 and 55).
//
// What becomes of a group's counts (PlanFor() chooses, with the figures):
//   few keys over many bins: another kernel, HistogramFewKeysKernel below.
//   one kernel (few bins, or few groups): the group adds its non-zero counters to the result itself, the 64
//       lanes of a wave to 64 neighbouring bins, each group from another place on because
//       atomics on ONE cache line retire at only ~0.1 G/s. Also above 2^28 keys, where the
//       partials would need more than 128 MiB of scratch, and when the scratch buffer cannot
//       be allocated.
//   two kernels (kMerge): the group stores a partial histogram of 65 KiB (less when n_bins is
//       below 16384; the words as they are, the copies of the warm counters summed) into a scratch
//       buffer, and a second kernel sums the partials column by column and adds the totals to
//       the result with one atomic per bin.
// The first version of this layout kept 16-bit halves for every bin and ballot counters for
// bins 0 and 1: partials of 128 KiB (32 MiB written and read back per 2^26 keys, now
// 16.25 MiB), 14 vector instructions per key (now 10), and LDS adds that serialised on the hot
// bins.
//
// Guard: entry check, and because a group has no side effects before its write-out,
// every wave re-reads the preempt word every kLoopKeys keys of the group (16384; a shorter chunk is checked
// at entry only) and the group abandons itself (its progress byte stays untagged, a replay redoes the chunk). The write-out
// runs to completion and commits. The groups of the merge kernel have progress bytes
// of their own behind those of the counting groups, and run only when every counting
// group has committed; the scratch buffer is the command's own from its first launch
// until it is destroyed, so the partials of a flushed launch are still there for the
// replay (a later command of the queue must not write into them: its groups may pass
// their entry check on a copy of the preempt word that has not been rewritten yet while
// this command is already flushed). Integer adds commute, so the result does not depend on the order in which work-groups (or
// replays) run.
#include <cmath>
#include <type_traits>

#include "hip_hal.h"
#include "xsched/hip/hal.h"

using namespace xsched::preempt;

namespace xsched::hip
{

namespace hist
{

constexpr uint32_t kThreads = 1024;
#ifndef XSCHED_HIST_UNITS
#define XSCHED_HIST_UNITS 1
#endif
constexpr uint32_t kUnits = XSCHED_HIST_UNITS;  // 128-bit loads per thread and iteration
#ifndef XSCHED_HIST_DEPTH
#define XSCHED_HIST_DEPTH 2
#endif
constexpr uint32_t kDepth = XSCHED_HIST_DEPTH;  // iterations of keys in flight or being counted
#ifndef XSCHED_HIST_POLL_TURNS
#define XSCHED_HIST_POLL_TURNS 2
#endif
constexpr uint32_t kPollTurns = XSCHED_HIST_POLL_TURNS; // turns of the ring per look at the preempt word
constexpr uint32_t kUnitKeys = kThreads * 4;
constexpr uint32_t kIterKeys = kUnitKeys * kUnits;
constexpr uint32_t kMinChunk = kUnitKeys;
constexpr uint32_t kMaxChunk = 1u << 18;
constexpr uint32_t kTargetGroups = 256;       // compute units of an MI355X
constexpr uint32_t kFewThreads = 256;         // HistogramFewKeysKernel: threads
constexpr uint32_t kFewKeys = kFewThreads * 4;        // keys per work-group
constexpr uint64_t kFewMaxKeys = 1u << 16;            // and the most keys it is used for
constexpr uint32_t kFewWarmBins = 256;                // its bins that are counted in order
constexpr uint32_t kColdWords = 1u << 14;           // word w counts bins w + i * 16384
constexpr uint32_t kWarmBins = 255;                 // bins below this have 32-bit counters of their own,
constexpr uint32_t kCopies = 16;                    // one per lane modulo 16
constexpr uint32_t kFewColdWords = 63u * 64;        // with at most this many cold words one per lane,
constexpr uint32_t kFewColdWarmBins = 256;          // and one bin more
constexpr uint32_t kOutside = 256;                  // counts a partial keeps outside the cold words (the last is 0 with more than kFewColdWords of them)
constexpr uint32_t kLdsBins = kColdWords + kWarmBins * kCopies;   // the cold words, then the warm counters
static_assert(kFewColdWords + kFewColdWarmBins * 64 <= kLdsBins && kFewColdWarmBins <= kOutside, "a warm counter per lane beside few cold words");
// The partial histograms of a launch in memory, n_part of them (one per counting group): the
// cold words column by column, one column per merge group, and within a column partial by
// partial: column c of partial p is the 64 words (256 bytes, two whole cache lines) at
// ((c * n_part) + p) * 64. A merge group therefore reads ONE contiguous run of n_part * 256
// bytes, and a counting group stores its partial as 256 pieces of two lines each. (Partial by
// partial, column by column inside, a merge group read 272 bytes out of every 68 KiB: three
// lines touched for two and a bit used, 1.41 times its bytes in traffic.) Behind the cold
// words: the counts of bins 0..255, which are kept outside them, partial by partial
// (1 KiB each). Columns that n_bins leaves empty are neither stored nor read.
constexpr uint32_t kMergeGroups = 256;
constexpr uint32_t kMergeThreads = 256;             // threads of a merge group
constexpr uint32_t kMergeWords = kColdWords / kMergeGroups;          // cold words per column (64)
constexpr uint32_t kPartialWords = kColdWords + kOutside;           // 65 KiB of scratch per counting group

/// Where column `column` of partial `p` lies, and where that partial's 256 outside counts do.
__host__ __device__ inline size_t ColumnAt(uint32_t column, uint32_t p, uint32_t n_part)
{
    return ((size_t)column * n_part + p) * kMergeWords;
}
__host__ __device__ inline size_t OutsideAt(uint32_t p, uint32_t n_part)
{
    return (size_t)n_part * kColdWords + (size_t)p * kOutside;
}
constexpr uint32_t kMaxPartials = 1024;
static_assert((uint64_t)kMaxPartials * kPartialWords * 4 < 0x7fffffffu, "a partial's stores have 31-bit offsets");
static_assert(kOutside == kMergeGroups && kWarmBins <= kOutside, "column j carries the outside count of bin j");
typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef i32x4 i32x4_any __attribute__((aligned(4)));   // keys may start at any int32

/// How many cold words n_bins bins use: whole columns.
__host__ __device__ inline uint32_t ColdWordsOf(uint32_t n_bins)
{
    return n_bins >= kColdWords ? kColdWords : (n_bins + kMergeWords - 1) / kMergeWords * kMergeWords;
}
/// log2 of a cold counter's bits; with at most 16384 bins nothing is ever shifted by it.
__host__ __device__ inline uint32_t ColdWidthLog2(uint32_t n_bins) { return n_bins > 2 * kColdWords ? 3 : 4; }

/// Keys per work-group for a histogram of n keys: a multiple of kMinChunk, at least
/// `floor` (rounded up to one).
inline uint32_t ChunkFor(uint64_t n, uint64_t floor = kMinChunk)
{
    uint64_t c = (n + kTargetGroups - 1) / kTargetGroups;
    if (c < floor) c = floor;
    c = (c + kMinChunk - 1) / kMinChunk * kMinChunk;
    if (c < kMinChunk) c = kMinChunk;
    if (c > kMaxChunk) c = kMaxChunk;
    return (uint32_t)c;
}

/// The least keys per work-group: a launch takes as long as its longest group (the more keys
/// the longer) plus what all groups together write out (the more groups the longer), which balances
/// where the keys of a group grow with the square root of all. Measured best: 2^18 keys 8192
/// (10.6 us; 16384: 10.8, 4096: 11.1), 2^20 16384 (12.1; 13.0, 13.4), 2^22 32768 to 65536 (16.5;
/// 16384: 17.5), and about the same with few bins (2^20 over 1000 bins: 8192 6.3 us, 16384 5.8,
/// 32768 6.5).
inline uint64_t ChunkFloor(uint64_t n) { return (uint64_t)(16.0 * std::sqrt((double)n)); }

enum class Way { kFew, kSweep, kMerge };

/// How n keys are counted (see the head of this file), in work-groups of `chunk` keys.
struct Plan { Way way; uint32_t chunk; uint64_t groups; };

/// LDS asked for on top of a counting group's own, so that it has its compute unit to itself.
/// Groups of long chunks may share one with another queue's (what one group does before its first
/// and behind its last key hides behind the other's keys: four queues of 2^26 keys 217 -> 208 us).
/// A launch of short ones is over before that pays, and two of its own groups on one unit while
/// others are free cost it more (2^20 and 2^22 keys: 1.0 us).
inline uint32_t ExtraLdsFor(uint32_t chunk) { return chunk < (1u << 17) ? 4096 : 0; }

/// - Few keys and many bins: HistogramFewKeysKernel. 16384 Zipf keys over 65536 bins take 3.8 us
///   (two kernels: 10.4), 65536 take 7.2, evenly spread 5.4 (10.5); 131072 take 11.8 (10.7).
/// - One kernel while the groups' sweeps are short, in wave-wide atomics of 64 neighbouring bins:
///   at most 768 per group (7 ns each; a whole 65536 bins is 1024: 12.5 us against 10.5 for two
///   kernels at 65536 keys), and 2^16 of all groups together (2^24 keys over 16000 bins, 2^16:
///   22.8 us against 23.8; over 20000 bins, 2^17: 28.8 against 24.6; over 1000 bins: 15.8
///   against 16.7; 2^18 keys over 1000 bins: 4.6 against 8.5).
/// - Two kernels otherwise.
inline Plan PlanFor(uint64_t n, uint32_t n_bins)
{
    if (n <= kFewMaxKeys && n_bins > kColdWords) return Plan { Way::kFew, kFewKeys, (n + kFewKeys - 1) / kFewKeys };
    const uint32_t chunk = ChunkFor(n, ChunkFloor(n));
    const uint64_t groups = (n + chunk - 1) / chunk;
    const uint64_t atomics = n_bins < kColdWords ? (n_bins + 63) / 64 : (uint64_t)((n_bins + kColdWords - 1) / kColdWords) * (kColdWords / 64);
    const bool sweep = (atomics <= 768 && groups * atomics <= (1u << 16)) || groups > kMaxPartials;
    return Plan { sweep ? Way::kSweep : Way::kMerge, chunk, groups };
}

struct Shared
{
    uint32_t bins[kLdsBins];
    uint32_t bailed;
    uint32_t guard_word;
    uint32_t invalid;       // keys outside [0, n_bins), absent ones included
    uint32_t sum;           // sum of all counters
    uint32_t runs;          // not 0: some wave saw runs of one key
    uint32_t least, most;   // a recount of such keys: the least and the largest
};
static_assert(sizeof(Shared) <= 80 * 1024, "two groups to a compute unit");

__device__ __forceinline__ void LdsAdd(uint32_t *p, uint32_t v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void GlobalAdd(uint32_t *p, uint32_t v)
{
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ void ClearBins(Shared &sh, uint32_t first, uint32_t end)
{
    for (uint32_t i = first + threadIdx.x * 4; i < end; i += kThreads * 4) *(u32x4 *)&sh.bins[i] = u32x4 { 0, 0, 0, 0 };
}

/// Where the warm counters of a launch lie: counter `copy` of bin b < bins is word first + (b << log2) + copy.
struct WarmPlace { uint32_t first, log2, bins; };
__device__ __forceinline__ WarmPlace WarmPlaceOf(uint32_t cold_words)
{
    static_assert(kCopies == 16, "log2 of it below");
    return cold_words <= kFewColdWords ? WarmPlace { kFewColdWords, 6, kFewColdWarmBins } : WarmPlace { kColdWords, 4, kWarmBins };
}

/// Where a valid key is counted, and by how much (see the head of this file); `copy` is the
/// lane's copy of warm bin 0.
template <bool kPacked>
__device__ __forceinline__ void SlotOf(uint32_t key, uint32_t copy, const WarmPlace &warm_at, uint32_t width_log2, uint32_t &word, uint32_t &inc)
{
    word = key < warm_at.bins ? copy + (key << warm_at.log2) : kPacked ? key & (kColdWords - 1) : key;
    inc = kPacked ? 1u << ((key >> 14) << width_log2) : 1u;
}

/// Sum of the counters (bytes or halves) of four cold words.
__device__ __forceinline__ uint32_t ColdSum(const u32x4 &w, bool bytes)
{
    if (!bytes) {
        return (w.x & 0xFFFFu) + (w.x >> 16) + (w.y & 0xFFFFu) + (w.y >> 16) + (w.z & 0xFFFFu) + (w.z >> 16) + (w.w & 0xFFFFu) + (w.w >> 16);
    }
    uint32_t sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_udot4(w[i], 0x01010101u, sum, false);
    return sum;
}

/// Stores of a partial, `at` bytes behind its launch's partials. They go through the L2 of the group's XCD to
/// memory (device scope, sc1): with plain stores the kernel ends by writing back what it left in
/// the L2s, and nothing else runs meanwhile. A launch of 2^20 / 2^22 / 14 million keys over 65536 bins and its merge
/// 10.9 / 15.2 / 23.0 us with those, 10.1 / 14.0 / 21.5 with these (9.6 / 11.7 / 16.2 if nothing were stored).
__device__ __forceinline__ void StorePartial(uint32_t *partials, size_t word, const u32x4 &w)
{
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(partials, 0, 0x7fffffff, 0x00020000);
    __builtin_amdgcn_raw_buffer_store_b128(w, r, (int)(uint32_t)(word * 4), 0, 0x10);
}
__device__ __forceinline__ void StorePartial(uint32_t *partials, size_t word, uint32_t w)
{
    __hip_atomic_store(partials + word, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t WaveSum(uint32_t v)
{
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

/// kPacked: a cold word holds the counters of two or four bins (n_bins above kColdWords). Where it is
/// one counter, the loop has no mask and no shift by a count from a register (2^22 even keys over 1000
/// bins 9.3 -> 8.0 us, 2^24 16.3 -> 14.0, 2^26 43.2 -> 40.5).
/// kMerge: the group stores its partial histogram (ColumnAt(), OutsideAt()) instead of adding its
/// counts to bins itself; HistogramMergeKernel does.
template <bool kGuard, bool kMerge, bool kPacked>
__global__ __launch_bounds__(kThreads, 8 /* waves per SIMD: two groups to a compute unit */)
void HistogramKernel(const int32_t *__restrict__ keys, uint64_t n, uint32_t *__restrict__ bins,
                     uint32_t n_bins, uint32_t chunk, uint32_t *__restrict__ partials, XGuardArgs g)
{
    __shared__ __attribute__((aligned(16))) Shared sh;

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t cold_words = ColdWordsOf(n_bins), width_log2 = ColdWidthLog2(n_bins);
    const XGuardBlock guard(g, blockIdx.x, &sh.guard_word);
    const XGuardEntry entry = kGuard ? guard.EnterBegin() : XGuardEntry {};   // on its way while the counters are cleared

    const WarmPlace warm_at = WarmPlaceOf(cold_words);
    const uint32_t copy = warm_at.first + (lane & ((1u << warm_at.log2) - 1u));
    ClearBins(sh, 0, cold_words);
    ClearBins(sh, warm_at.first, warm_at.first + (warm_at.bins << warm_at.log2));
    if (tid == 0) { sh.bailed = 0; sh.invalid = 0; sh.sum = 0; sh.runs = 0; sh.least = ~0u; sh.most = 0; }

    const uint64_t begin = (uint64_t)blockIdx.x * chunk;
    const uint64_t end = begin + chunk < n ? begin + chunk : n;
    const uint64_t full_end = begin + (end - begin) / kIterKeys * kIterKeys;

    // 128-bit loads whatever the array's alignment: a global load takes any multiple of four bytes.
    auto load_iter = [&](i32x4 *v, uint64_t base) {
#pragma unroll
        for (uint32_t u = 0; u < kUnits; ++u) {
            v[u] = __builtin_nontemporal_load((const i32x4_any *)(keys + base + ((uint64_t)u * kThreads + tid) * 4));
            if (u + 1 < kUnits) asm volatile("" ::: "memory");
        }
    };
    // A ring of kDepth register sets: the set just counted is refilled with the keys of
    // kDepth iterations ahead. The first sets are requested before the guard's decision
    // (reading keys has no side effect).
    constexpr uint64_t kTurnKeys = (uint64_t)kDepth * kIterKeys;
    constexpr uint64_t kLoopKeys = kTurnKeys * kPollTurns; // one trip of the main loop
    const uint64_t turns_end = begin + (full_end - begin) / kLoopKeys * kLoopKeys;
    i32x4 ring[kDepth][kUnits];
    if (begin < turns_end) {
        // Every set is loaded, no branch per set, and in the order in which the loop
        // refills them (the empty statements keep the scheduler from permuting the loads:
        // the loop's waits count on that order). A chunk shorter than one trip of the loop
        // does not use it at all, so that these registers are written on this path only.
#pragma unroll
        for (uint32_t d = 0; d < kDepth; ++d) {
            load_iter(ring[d], begin + (uint64_t)d * kIterKeys);
            asm volatile("" ::: "memory");
        }
    }

    if (kGuard) {
        if (!guard.EnterEnd(entry)) return; // contains the barrier that also publishes the cleared counters
    } else {
        __syncthreads();
    }

    uint32_t invalid = 0; // keys of this thread outside [0, n_bins), absent ones included

    // Whether the wave's keys look like runs of one key (sorted or constant keys): asked of the first
    // of a chunk that is long enough for the main loop. (Three lanes in four, which the hottest key of a
    // skewed distribution does not reach. Asked in every iteration, of short chunks or where a word is one
    // counter it costs a launch 0.2-0.4 us.)
    bool runs = false;
    auto look_for_runs = [&](const i32x4 &v) { runs = kPacked && __popcll(__ballot(v.x == v.w)) >= 48; };

    // Counts kUnitsNow * 4 keys per thread.
    auto process = [&](const i32x4 *v, auto units_tag) {
        constexpr uint32_t kN = decltype(units_tag)::value * 4;
        uint32_t k[kN];
#pragma unroll
        for (uint32_t u = 0; u < kN / 4; ++u) {
            k[u * 4 + 0] = (uint32_t)v[u].x; k[u * 4 + 1] = (uint32_t)v[u].y;
            k[u * 4 + 2] = (uint32_t)v[u].z; k[u * 4 + 3] = (uint32_t)v[u].w;
        }
        // Are all keys of the wave below n_bins (the usual case)? One max per key and one
        // vote per iteration decide it; then nothing has to be tallied per key and the
        // LDS add needs no branch.
        uint32_t largest = k[0];
#pragma unroll
        for (uint32_t j = 1; j < kN; ++j) largest = largest > k[j] ? largest : k[j];
        if (__ballot(largest >= n_bins) == 0 && !runs) {
#pragma unroll
            for (uint32_t j = 0; j < kN; ++j) {
                uint32_t word, inc;
                SlotOf<kPacked>(k[j], copy, warm_at, width_log2, word, inc);
                LdsAdd(&sh.bins[word], inc);
            }
        } else {
            // A thread whose keys are all the same adds them at once: a quarter of the adds that
            // meet on one address.
            bool same = true;
#pragma unroll
            for (uint32_t j = 1; j < kN; ++j) same = same && k[j] == k[0];
            const uint32_t times = same ? kN : 1u;
#pragma unroll
            for (uint32_t j = 0; j < kN; ++j) {
                if (j != 0 && same) continue;
                if (k[j] >= n_bins) {
                    invalid += times;
                } else {
                    uint32_t word, inc;
                    SlotOf<kPacked>(k[j], copy, warm_at, width_log2, word, inc);
                    LdsAdd(&sh.bins[word], inc * times);
                }
            }
        }
    };
    using Units = std::integral_constant<uint32_t, kUnits>;
    using OneUnit = std::integral_constant<uint32_t, 1>;

    // Counts the chunk; false when the wave saw a deactivation and gave up.
    //
    // Full iterations go through the ring. Whole turns of it run without a branch around
    // their loads (a refill that would start beyond the last full iteration re-reads that
    // one instead, unused), so the compiler can count exactly how many loads may still be
    // in flight where it needs one of them. The preempt word is requested at the start of
    // a trip of the loop (kPollTurns turns) and looked at at its end: by then the refills
    // issued behind it are the only loads it does not wait for.
    auto count_chunk = [&]() -> bool {
        uint64_t base = begin;
        if (base < turns_end) {
            look_for_runs(ring[0][0]);
            do {
                const uint32_t polled = kGuard ? guard.WavePollBegin() : 0u;
#pragma unroll
                for (uint32_t t = 0; t < kPollTurns; ++t) {
#pragma unroll
                    for (uint32_t d = 0; d < kDepth; ++d) {
                        process(ring[d], Units {});
                        const uint64_t next = base + (uint64_t)d * kIterKeys + kTurnKeys;
                        load_iter(ring[d], next < full_end ? next : full_end - kIterKeys);
                    }
                    base += kTurnKeys;
                }
                if (kGuard && !guard.WavePollEnd(polled)) return false;
            } while (base < turns_end);
            // fewer than kDepth full iterations are left, and their keys are in the ring already
#pragma unroll
            for (uint32_t d = 0; d < kDepth; ++d) {
                if (base < full_end) {
                    process(ring[d], Units {});
                    base += kIterKeys;
                }
            }
        }
        // what a chunk has beyond whole trips of the loop and the ring: one iteration at a time
        for (; base < full_end; base += kIterKeys) {
            i32x4 v[kUnits];
            load_iter(v, base);
            process(v, Units {});
        }
        // Ragged remainder: one unit at a time, absent keys read as the sentinel.
        for (; base < end; base += kUnitKeys) {
            const uint64_t idx = base + (uint64_t)tid * 4;
            i32x4 v = { -1, -1, -1, -1 };
            if (idx + 3 < end) {
                v = __builtin_nontemporal_load((const i32x4_any *)(keys + idx));
            } else {
                if (idx + 0 < end) v.x = keys[idx + 0];
                if (idx + 1 < end) v.y = keys[idx + 1];
                if (idx + 2 < end) v.z = keys[idx + 2];
                if (idx + 3 < end) v.w = keys[idx + 3];
            }
            process(&v, OneUnit {});
        }
        return true;
    };
    if (!count_chunk() && lane == 0) sh.bailed = 1;
    if (kPacked && runs && lane == 0) sh.runs = 1;

    // One LDS add per wave: in the group with the ragged end nearly every lane has absent keys, and 1024 lanes
    // that add to this one address took 3 us of nearly every launch (2^17 + 77 keys over 1000 bins 18.5 -> 15.4 us a pass).
    if (__ballot(invalid != 0) != 0) {
        invalid = WaveSum(invalid);
        if (lane == 0) LdsAdd(&sh.invalid, invalid);
    }
    __syncthreads();

    if (kGuard) {
        // Last point without side effects: the group abandons if any of its waves saw a
        // deactivation (the barrier above published their verdicts). The preempt word is
        // not read again here: that round trip would sit exposed in front of every
        // write-out, and a group that writes out just after a deactivation is no different
        // from one that was a little further along.
        if (sh.bailed != 0) return;
    }

    const uint32_t me = blockIdx.x, n_part = gridDim.x;
    uint32_t counted = 0;
    // the copies of warm bin tid / 4: four threads sum a quarter each
    uint32_t warm = 0;
    if (tid / 4 < warm_at.bins) {
        for (uint32_t q = 0; q < 1u << (warm_at.log2 - 4); ++q) {
            const u32x4 w = *(const u32x4 *)&sh.bins[warm_at.first + ((tid * 4) << (warm_at.log2 - 4)) + q * 4];
            warm += w.x + w.y + w.z + w.w;
        }
    }
    counted += warm;
    warm += __shfl_xor(warm, 1);
    warm += __shfl_xor(warm, 2);
    if (kMerge) {
        // Every group starts at a column of its own: column c of all partials is one run of
        // n_part * 256 bytes, and groups that all wrote column 0 first, then column 1, would
        // all be storing into the same few DRAM pages at any moment.
        const uint32_t turn = me * 37u % (cold_words / kMergeWords) * kMergeWords;
        for (uint32_t k = tid * 4; k < cold_words; k += kThreads * 4) {
            const uint32_t i = k + turn < cold_words ? k + turn : k + turn - cold_words;
            const u32x4 w = *(const u32x4 *)&sh.bins[i];
            StorePartial(partials, ColumnAt(i / kMergeWords, me, n_part) + i % kMergeWords, w);
            if (kPacked) counted += ColdSum(w, width_log2 == 3);
        }
        if (tid % 4 == 0) StorePartial(partials, OutsideAt(me, n_part) + tid / 4, warm);
    } else if (kPacked) {
        for (uint32_t k = tid * 4; k < cold_words; k += kThreads * 4) counted += ColdSum(*(const u32x4 *)&sh.bins[k], width_log2 == 3);
    }

    bool exact = true;
    if (kPacked) {
        // One LDS add per wave: 1024 lanes adding to this one address took 3.4 us of every launch.
        counted = WaveSum(counted);
        if (lane == 0) LdsAdd(&sh.sum, counted);
        __syncthreads();
        // every key slot the group went through (absent keys of the ragged end included) is
        // an invalid key or in the counters
        const uint32_t expected = (uint32_t)(full_end - begin)
                                + (uint32_t)((end - full_end + kUnitKeys - 1) / kUnitKeys) * kUnitKeys - sh.invalid;
        exact = __builtin_amdgcn_readfirstlane(sh.sum) == __builtin_amdgcn_readfirstlane(expected);
    }
    if (!exact) {
        // A counter overflowed: this group's partial counts nothing, and the chunk is counted
        // again with 32-bit counters, one quarter of the bins at a time.
        __syncthreads();
        if (kMerge) {
            for (uint32_t i = tid * 4; i < cold_words; i += kThreads * 4) {
                StorePartial(partials, ColumnAt(i / kMergeWords, me, n_part) + i % kMergeWords, u32x4 { 0, 0, 0, 0 });
            }
            if (tid < kOutside) StorePartial(partials, OutsideAt(me, n_part) + tid, 0u);
        }
        // Runs of one key are added a thread's four at a time, as above, and the first pass finds
        // the least and the largest key: quarters outside them are passed over. (Keys without runs
        // gain nothing by either, and the questions are 1 us of each pass.)
        auto recount = [&](auto of_runs) {
            constexpr bool kRuns = decltype(of_runs)::value;
            for (uint32_t first = 0; first < n_bins; first += kColdWords) {
                const uint32_t count = n_bins - first < kColdWords ? n_bins - first : kColdWords;
                if (kRuns && first != 0 && (sh.most < first || sh.least >= first + kColdWords)) continue;   // the same for the whole group
                ClearBins(sh, 0, kColdWords);
                __syncthreads();
                uint32_t least = ~0u, most = 0;
                auto add = [&](const i32x4 &v) {
                    const bool same = kRuns && v.x == v.y && v.x == v.z && v.x == v.w;
#pragma unroll
                    for (uint32_t j = 0; j < 4; ++j) {
                        const uint32_t key = (uint32_t)v[j];
                        if ((j == 0 || !same) && key - first < count) LdsAdd(&sh.bins[key - first], same ? 4u : 1u);
                        if (kRuns && first == 0) {
                            least = least < key ? least : key;
                            most = most > key ? most : key;   // (a key outside the bins is larger than all: no quarter is passed over then)
                        }
                    }
                };
                uint64_t base = begin;
                auto add_units = [&](auto at_once) {   // loads in flight per thread
                    constexpr uint32_t kAtOnce = decltype(at_once)::value;
                    for (; base + kAtOnce * kUnitKeys <= end; base += kAtOnce * kUnitKeys) {
                        i32x4 v[kAtOnce];
#pragma unroll
                        for (uint32_t u = 0; u < kAtOnce; ++u) v[u] = *(const i32x4_any *)(keys + base + u * kUnitKeys + (uint64_t)tid * 4);
#pragma unroll
                        for (uint32_t u = 0; u < kAtOnce; ++u) add(v[u]);
                    }
                };
                add_units(std::integral_constant<uint32_t, 4> {});
                add_units(std::integral_constant<uint32_t, 2> {});   // (a chunk of the least size)
                for (; base < end; base += kUnitKeys) {
                    const uint64_t idx = base + (uint64_t)tid * 4;
                    i32x4 v = { -1, -1, -1, -1 };
                    if (idx + 3 < end) {
                        v = *(const i32x4_any *)(keys + idx);
                    } else {
                        if (idx + 0 < end) v.x = keys[idx + 0];
                        if (idx + 1 < end) v.y = keys[idx + 1];
                        if (idx + 2 < end) v.z = keys[idx + 2];
                    }
                    add(v);
                }
                if (kRuns && first == 0) {
                    // (per wave first, like the sum above)
#pragma unroll
                    for (int d = 32; d > 0; d >>= 1) {
                        const uint32_t l = __shfl_xor(least, d), m = __shfl_xor(most, d);
                        least = least < l ? least : l;
                        most = most > m ? most : m;
                    }
                    if (lane == 0) {
                        __hip_atomic_fetch_min(&sh.least, least, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                        __hip_atomic_fetch_max(&sh.most, most, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    }
                }
                __syncthreads();
                for (uint32_t k = tid; k < kColdWords; k += kThreads) {
                    const uint32_t i = (k + me * 2368u) % kColdWords;   // another line for every group
                    const uint32_t c = sh.bins[i];
                    if (c != 0) GlobalAdd(bins + first + i, c);
                }
                __syncthreads();
            }
        };
        if (__builtin_amdgcn_readfirstlane(sh.runs) != 0) recount(std::true_type {});
        else recount(std::false_type {});
    } else if (!kMerge) {
        const uint32_t turn = me * 37u % (cold_words / kMergeWords) * kMergeWords;
        auto sweep = [&](auto counters_per_word) {
            constexpr uint32_t kCounters = decltype(counters_per_word)::value, kWidth = 32 / kCounters;
#pragma unroll 4
            for (uint32_t k = tid; k < cold_words; k += kThreads) {
                const uint32_t i = k + turn < cold_words ? k + turn : k + turn - cold_words;
                const uint32_t w = sh.bins[i];
#pragma unroll
                for (uint32_t c = 0; c < kCounters; ++c) {
                    const uint32_t count = kCounters == 1 ? w : w >> (c * kWidth) & ((1u << (kWidth & 31)) - 1u);
                    if (count != 0) GlobalAdd(bins + i + c * kColdWords, count);
                }
            }
        };
        if (!kPacked) sweep(std::integral_constant<uint32_t, 1> {});
        else if (width_log2 == 4) sweep(std::integral_constant<uint32_t, 2> {});
        else sweep(std::integral_constant<uint32_t, 4> {});
        if (tid % 4 == 0 && warm != 0) GlobalAdd(bins + tid / 4, warm);   // counts of bins that n_bins ends before are 0
    }

    if (kGuard) guard.Commit();
}

using CountKernelFn = void (*)(const int32_t *, uint64_t, uint32_t *, uint32_t, uint32_t, uint32_t *, XGuardArgs);
template <bool kMerge>
inline CountKernelFn CountKernel(bool guarded, uint32_t n_bins)
{
    if (n_bins > kColdWords) return guarded ? HistogramKernel<true, kMerge, true> : HistogramKernel<false, kMerge, true>;
    return guarded ? HistogramKernel<true, kMerge, false> : HistogramKernel<false, kMerge, false>;
}

/// Few keys, many bins: a group of 256 threads has 1024 keys, four to a thread. Bins below 256 are
/// counted in LDS and added to the result by the group's threads in order, one line-wide atomic
/// per sixteen of them (these are the bins that every group has, and atomics on one line retire
/// one after the other). Of the other counters (16 bits per bin: word k & 32767, half k >> 15;
/// 1024 keys cannot overflow one) a group touches only the words of its own keys: each thread
/// zeroes its four, then all count, then each takes what is in its four out again with one
/// atomic that leaves zero behind, so of all threads that hold a key exactly one gets its count
/// and adds it to the result. Nothing is cleared and nothing swept: with few keys to a group, the
/// sweep over 65536 counters is 1024 wave-wide atomics with a lane or two in each (7 us).
template <bool kGuard>
__global__ __launch_bounds__(kFewThreads)
void HistogramFewKeysKernel(const int32_t *__restrict__ keys, uint64_t n, uint32_t *__restrict__ bins,
                            uint32_t n_bins, XGuardArgs g)
{
    __shared__ uint32_t halves[1u << 15];
    __shared__ uint32_t warm[kFewWarmBins];
    __shared__ uint32_t guard_word;
    static_assert(kFewThreads == kFewWarmBins, "a thread per warm bin");

    const XGuardBlock guard(g, blockIdx.x, &guard_word);
    const XGuardEntry entry = kGuard ? guard.EnterBegin() : XGuardEntry {};
    const uint32_t tid = threadIdx.x;
    const uint64_t idx = (uint64_t)blockIdx.x * kFewKeys + (uint64_t)tid * 4;
    i32x4 v = { -1, -1, -1, -1 };
    if (idx + 3 < n) {
        v = __builtin_nontemporal_load((const i32x4_any *)(keys + idx));
    } else {
        if (idx + 0 < n) v.x = keys[idx + 0];
        if (idx + 1 < n) v.y = keys[idx + 1];
        if (idx + 2 < n) v.z = keys[idx + 2];
    }
    warm[tid] = 0;
    if (kGuard && !guard.EnterEnd(entry)) return;

    const uint32_t k[4] = { (uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w };
    const uint32_t cold_bins = n_bins > kFewWarmBins ? n_bins - kFewWarmBins : 0;   // k - kFewWarmBins < cold_bins: a cold key
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) if (k[j] - kFewWarmBins < cold_bins) halves[k[j] & 0x7FFFu] = 0;
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        if (k[j] - kFewWarmBins < cold_bins) LdsAdd(&halves[k[j] & 0x7FFFu], 1u << (k[j] >> 15) * 16);
        else if (k[j] < n_bins) LdsAdd(&warm[k[j]], 1u);
    }
    __syncthreads();
    uint32_t count[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
        count[j] = 0;
        if (k[j] - kFewWarmBins >= cold_bins) continue;
        const uint32_t shift = (k[j] >> 15) * 16;
        const uint32_t old = __hip_atomic_fetch_and(&halves[k[j] & 0x7FFFu], ~(0xFFFFu << shift), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        count[j] = old >> shift & 0xFFFFu;
    }
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) if (count[j] != 0) GlobalAdd(bins + k[j], count[j]);
    if (warm[tid] != 0) GlobalAdd(bins + tid, warm[tid]);
    if (kGuard) guard.Commit();
}

/// Sums the partial histograms of the counting groups and adds the totals to bins. Group j
/// owns column j of every partial: 64 cold words (counter i of word w = bin w + i * 16384; a
/// byte, a half or the whole word each) if n_bins reaches that far, and the count of bin j,
/// which is kept outside them. Thread (row, col)
/// reads four cold words of its column from partials row, row + 16, ... (the sixteen threads
/// of a row one partial's 256 bytes, the four rows of a wave four neighbouring partials: one
/// KiB in a piece); the threads of col 0 also read the outside count. The group's progress
/// byte is first_wg + j. Four waves per group: the kernel is one round trip to its partials,
/// a reduction through 16 KiB of LDS and 256 atomics.
template <bool kGuard>
__global__ __launch_bounds__(kMergeThreads)
void HistogramMergeKernel(const uint32_t *__restrict__ partials, uint32_t n_part, uint32_t *__restrict__ bins,
                          uint32_t n_bins, uint32_t first_wg, XGuardArgs g)
{
    constexpr uint32_t kCols = kMergeWords / 4, kRows = kMergeThreads / kCols; // 16 x 16
    constexpr uint32_t kAhead = 16;                                      // rows requested before the guard's reads
    __shared__ uint32_t red[kRows][16][kCols];   // per row: the 16 counters of each of the 16 word quads
    __shared__ uint32_t total[16][kCols];
    __shared__ uint32_t outside_total;
    __shared__ uint32_t guard_word;

    const uint32_t tid = threadIdx.x;
    const uint32_t col = tid % kCols, row = tid / kCols;
    const uint32_t column = blockIdx.x;
    const bool has_column = column * kMergeWords < ColdWordsOf(n_bins);
    const bool bytes = n_bins > 2 * kColdWords, halves = n_bins > kColdWords;
    const uint32_t even_mask = bytes ? 0x00FF00FFu : halves ? 0xFFFFu : 0xFFFFFFFFu;
    const uint32_t odd_mask = halves ? even_mask : 0u, odd_shift = bytes ? 8u : 16u;
    auto load_words = [&](uint32_t p) {
        return has_column && p < n_part ? *(const u32x4 *)(partials + ColumnAt(column, p, n_part) + col * 4) : u32x4 { 0, 0, 0, 0 };
    };
    auto load_outside = [&](uint32_t p) {
        return col == 0 && p < n_part ? partials[OutsideAt(p, n_part) + column] : 0u;
    };
    // even[i] holds bytes 0 and 2 of word i in its halves, odd[i] bytes 1 and 3 (a thread adds
    // at most kMaxPartials / kRows = 64 values of 255 into a half); or half 0 and half 1; or the
    // whole word and nothing.
    uint32_t even[4] = { 0, 0, 0, 0 }, odd[4] = { 0, 0, 0, 0 }, outside = 0;
    auto add_words = [&](const u32x4 &w) {
        const uint32_t v[4] = { w.x, w.y, w.z, w.w };
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) { even[i] += v[i] & even_mask; odd[i] += (v[i] >> odd_shift) & odd_mask; }
    };
    // The first rows are requested before the guard's reads: the kernel is short, and the
    // round trips overlap. Reading has no side effect (after a flushed counting launch the
    // words are stale, and nothing is done with them).
    u32x4 first[kAhead];
    uint32_t first_outside[kAhead];
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) {
        first[i] = load_words(row + i * kRows);
        first_outside[i] = load_outside(row + i * kRows);
    }
    if (tid == 0) {
        outside_total = 0;
        // This kernel does not look at the preempt word itself: it runs for a few
        // microseconds, and what it must not do is run after a counting launch that was
        // flushed, whose partials are incomplete. Every counting group that leaves because of
        // a deactivation puts the epoch of its launch into the `flushed` word before it does
        // (and every group that starts later finds the word and leaves the same way): the
        // word differs from this launch's epoch exactly when every counting group has run to
        // its end, now or in an earlier launch. The group's own tag says whether it has added
        // its column already, before a flush that made this launch a replay.
        bool go = true;
        if (kGuard) {
            go = !xguard_epoch_flushed(g);
            if (go && g.resume && g.done && xguard_committed(g, first_wg + blockIdx.x)) go = false;
        }
        guard_word = go ? 1u : 0u;
    }
    __syncthreads();
    if (kGuard && guard_word == 0) return;

#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) { add_words(first[i]); outside += first_outside[i]; }
#pragma unroll 4
    for (uint32_t p = row + kAhead * kRows; p < n_part; p += kRows) { add_words(load_words(p)); outside += load_outside(p); }
    // counter b * 4 + i of a thread: counter b of its word i
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
        red[row][0 + i][col] = bytes ? even[i] & 0xFFFFu : even[i];
        red[row][4 + i][col] = bytes ? odd[i] & 0xFFFFu : odd[i];
        red[row][8 + i][col] = bytes ? even[i] >> 16 : 0u;
        red[row][12 + i][col] = bytes ? odd[i] >> 16 : 0u;
    }
    if (outside != 0) LdsAdd(&outside_total, outside);
    __syncthreads();
    static_assert(kMergeThreads == 16 * kCols, "one thread per counter of the column");
    {
        const uint32_t v = tid / kCols, c = tid % kCols;
        uint32_t t = 0;
#pragma unroll 16
        for (uint32_t r = 0; r < kRows; ++r) t += red[r][v][c];
        total[v][c] = t;
    }
    __syncthreads();

    // 256 counters: counter (b, i) of quad c is bin column * 64 + c * 4 + i + b * 16384. One
    // 32-bit add each, nothing returned, so no wave waits for the round trip; the 64 lanes of a
    // wave add to 64 neighbouring bins.
    {
        const uint32_t b = tid / 64, c = (tid % 64) / 4, i = tid % 4;
        const uint32_t count = total[b * 4 + i][c];
        const uint32_t bin = column * kMergeWords + c * 4 + i + b * kColdWords;
        if (count != 0 && bin < n_bins) GlobalAdd(bins + bin, count);
    }
    if (tid == 0) {
        // bin <column>, counted outside the cold words (which hold nothing for bins below 255; bin 255
        // has its count in one of the two and 0 in the other)
        if (outside_total != 0 && column < n_bins) GlobalAdd(bins + column, outside_total);
    }
    if (kGuard) {
        XGuardBlock guard(g, first_wg + blockIdx.x, &guard_word);
        guard.Commit();
    }
}

class HipHistogramCommand final : public HipGuardedCommand
{
public:
    /// plan.groups counting groups; with two kernels, kMergeGroups merge groups follow them in
    /// the progress map.
    HipHistogramCommand(const void *keys, size_t n, void *bins, uint32_t n_bins, const Plan &plan, int guard_mode)
        : HipGuardedCommand((uint32_t)plan.groups + (plan.way == Way::kMerge ? kMergeGroups : 0), guard_mode)
        , keys_((const int32_t *)keys), n_(n), bins_((uint32_t *)bins), n_bins_(n_bins), chunk_(plan.chunk)
        , n_count_wg_((uint32_t)plan.groups), way_(plan.way) {}
    virtual ~HipHistogramCommand() { if (partials_ != nullptr) pool_->Release(partials_); }

protected:
    size_t ScratchBytes() const { return (size_t)n_count_wg_ * kPartialWords * sizeof(uint32_t); }

    virtual void ReserveOnSubmit(HipQueue &q) override
    {
        if (way_ == Way::kMerge && n_ != 0 && partials_ == nullptr) q.Scratch()->Reserve(ScratchBytes());
    }

    virtual hipError_t PrepareLaunch(HipQueue &q) override
    {
        // A replay must find the partials of the flushed launch: the buffer taken at the
        // first launch is kept until the command is destroyed.
        if (way_ != Way::kMerge || n_ == 0 || partials_ != nullptr) return hipSuccess;
        pool_ = q.Scratch();
        partials_ = (uint32_t *)pool_->Acquire(ScratchBytes());
        // No scratch: one kernel works on the same chunks (decided before the first launch,
        // so every replay takes the same path).
        if (partials_ == nullptr) way_ = Way::kSweep;
        return hipSuccess;
    }

    virtual hipError_t LaunchKernel(hipStream_t stream, bool guarded, const XGuardArgs &g) override
    {
        if (n_ == 0) return hipSuccess;
        const dim3 grid(n_count_wg_), block(kThreads);
        if (way_ == Way::kFew) {
            LaunchWithStop(TakeStopEvent(), guarded ? HistogramFewKeysKernel<true> : HistogramFewKeysKernel<false>, grid, dim3(kFewThreads), stream,
                           keys_, (uint64_t)n_, bins_, n_bins_, g);
            return hipGetLastError();
        }
        if (way_ == Way::kSweep) {
            LaunchWithStopLds(ExtraLdsFor(chunk_), TakeStopEvent(), CountKernel<false>(guarded, n_bins_), grid, block, stream,
                           keys_, (uint64_t)n_, bins_, n_bins_, chunk_, (uint32_t *)nullptr, g);
            return hipGetLastError();
        }
        // the merge kernel is the command's last
        LaunchWithStopLds(ExtraLdsFor(chunk_), nullptr, CountKernel<true>(guarded, n_bins_), grid, block, stream,
                       keys_, (uint64_t)n_, bins_, n_bins_, chunk_, partials_, g);
        hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        LaunchWithStop(TakeStopEvent(), guarded ? HistogramMergeKernel<true> : HistogramMergeKernel<false>, dim3(kMergeGroups), dim3(kMergeThreads), stream,
                       (const uint32_t *)partials_, n_count_wg_, bins_, n_bins_, n_count_wg_, g);
        return hipGetLastError();
    }

private:
    const int32_t *keys_;
    const size_t n_;
    uint32_t *bins_;
    const uint32_t n_bins_;
    const uint32_t chunk_;
    const uint32_t n_count_wg_;
    Way way_;
    std::shared_ptr<ScratchPool> pool_;
    uint32_t *partials_ = nullptr;
};

} // namespace hist

} // namespace xsched::hip

using namespace xsched::hip;

// ---- the entry point that allocates nothing -------------------------------------------
//
// The partial histograms of HipHistogramLaunchNoAlloc() live in this array instead of a
// buffer from a queue's pool. Every GPU the library runs on holds its own copy at its own
// address for the life of the process; in host code the array's NAME is only a handle for
// hipGetSymbolAddress(), never a device pointer.
namespace
{
constexpr uint32_t kNoAllocMaxGroups = 256;                       // counting work-groups
constexpr uint64_t kNoAllocMaxKeys = (uint64_t)kNoAllocMaxGroups * hist::kMaxChunk; // 2^26
constexpr size_t kNoAllocScratchWords = (size_t)kNoAllocMaxGroups * hist::kPartialWords;

static __device__ __align__(256) uint32_t scratch[kNoAllocScratchWords];          // 16.25 MiB

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_scratch_mtx;
uint32_t *g_scratch_ptr[kNoAllocMaxDevices] = {};

/// Device address of `scratch` on `device`, which must be the calling thread's current device.
/// Looked up once per device (when a hardware queue is created there, else at the entry
/// point's first call on it); nullptr (and a warning) if the runtime refuses. The first
/// lookup may load the code object, which allocates: it runs with the thread's capture mode
/// relaxed, so a capture under way on ANOTHER stream is not invalidated by it, but it cannot
/// be part of a capture itself: the first call on a device comes before the capture begins.
uint32_t *ScratchOnCurrentDevice(int device)
{
    if (device < 0 || device >= kNoAllocMaxDevices) return nullptr;
    std::lock_guard<std::mutex> lock(g_scratch_mtx);
    if (g_scratch_ptr[device] != nullptr) return g_scratch_ptr[device];
    RelaxedCaptureScope relaxed;
    uint32_t *ptr = nullptr;
    const hipError_t err = hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch));
    if (err != hipSuccess || ptr == nullptr) {
        XWARN("hipGetSymbolAddress(scratch) on device %d failed: %d (%s)", device, (int)err, hipGetErrorString(err));
        (void)hipGetLastError();
        return nullptr;
    }
    g_scratch_ptr[device] = ptr;
    return ptr;
}
} // namespace

namespace xsched::hip
{
bool ResolveNoAllocScratch(int device) { return ScratchOnCurrentDevice(device) != nullptr; }
} // namespace xsched::hip

EXPORT_C_FUNC XResult HipHistogramLaunchNoAlloc(void *stream_ptr, const void *keys, size_t n, void *bins,
                                                uint32_t n_bins)
{
    if (bins == nullptr || (n != 0 && keys == nullptr)) return kXSchedErrorInvalidValue;
    if (n_bins == 0 || n_bins > 65536) return kXSchedErrorInvalidValue;
    if (n > kNoAllocMaxKeys) {
        XWARN("HipHistogramLaunchNoAlloc: %zu keys exceed the limit of %llu keys that the static "
              "scratch array holds partial histograms for", n, (unsigned long long)kNoAllocMaxKeys);
        return kXSchedErrorInvalidValue;
    }
    if (n == 0) return kXSchedSuccess;

    hipStream_t stream = (hipStream_t)stream_ptr;
    int device = -1, current = -1;
    if (hipGetDevice(&current) != hipSuccess) return kXSchedErrorHardware;
    if (stream == nullptr) device = current;
    else if (hipStreamGetDevice(stream, &device) != hipSuccess) { (void)hipGetLastError(); return kXSchedErrorInvalidValue; }
    if (device < 0 || device >= kNoAllocMaxDevices) return kXSchedErrorNotSupported;
    // Symbol lookup and launch both act on the current device: it has to be the stream's.
    if (device != current && hipSetDevice(device) != hipSuccess) return kXSchedErrorHardware;

    XResult res = kXSchedSuccess;
    uint32_t *partials = ScratchOnCurrentDevice(device);
    if (partials == nullptr) {
        res = kXSchedErrorHardware;
    } else {
        // Every group of the two-kernel way stores its complete partial (all-zero after an
        // overflow recount), so nothing of an earlier call's contents is read and nothing has to
        // be cleared.
        const hist::Plan plan = hist::PlanFor(n, n_bins);   // its chunks grow with n: at most 256 groups up to 2^26 keys
        XASSERT(plan.groups <= kNoAllocMaxGroups && plan.chunk <= hist::kMaxChunk, "group count %llu / chunk %u out of range",
                (unsigned long long)plan.groups, plan.chunk);
        const XGuardArgs inert {};
        const dim3 grid((uint32_t)plan.groups), block(hist::kThreads);
        const int32_t *const k = (const int32_t *)keys;
        uint32_t *const out = (uint32_t *)bins;
        if (plan.way == hist::Way::kFew) {
            hipLaunchKernelGGL(hist::HistogramFewKeysKernel<false>, grid, dim3(hist::kFewThreads), 0, stream, k, (uint64_t)n, out, n_bins, inert);
        } else if (plan.way == hist::Way::kSweep) {
            hipLaunchKernelGGL(hist::CountKernel<false>(false, n_bins), grid, block, hist::ExtraLdsFor(plan.chunk), stream, k, (uint64_t)n, out, n_bins, plan.chunk,
                               (uint32_t *)nullptr, inert);
        } else {
            hipLaunchKernelGGL(hist::CountKernel<true>(false, n_bins), grid, block, hist::ExtraLdsFor(plan.chunk), stream, k, (uint64_t)n, out, n_bins, plan.chunk, partials, inert);
            if (hipGetLastError() == hipSuccess) {
                hipLaunchKernelGGL(hist::HistogramMergeKernel<false>, dim3(hist::kMergeGroups), dim3(hist::kMergeThreads), 0, stream,
                                   (const uint32_t *)partials, (uint32_t)plan.groups, out, n_bins, (uint32_t)plan.groups, inert);
            }
        }
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) {
            XWARN("HipHistogramLaunchNoAlloc: launch failed: %d (%s)", (int)err, hipGetErrorString(err));
            res = kXSchedErrorHardware;
        }
    }
    if (device != current) (void)hipSetDevice(current);
    return res;
}

EXPORT_C_FUNC XResult HipHistogramCommandCreate(HwCommandHandle *cmd, const void *keys, size_t n,
                                                void *bins, uint32_t n_bins, int guard)
{
    if (cmd == nullptr || bins == nullptr || (n != 0 && keys == nullptr) || guard < 0 || guard > 3) {
        return kXSchedErrorInvalidValue;
    }
    if (n_bins == 0 || n_bins > 65536) return kXSchedErrorInvalidValue;
    hist::Plan plan = hist::PlanFor(n == 0 ? 1 : n, n_bins);
    // Two variables take the choice over: the number of keys from which two kernels are used
    // (one kernel below it), and the least keys per work-group.
    const char *min_keys = getenv("XSCHED_HIP_HIST_MERGE_MIN_KEYS"), *floor = getenv("XSCHED_HIP_HIST_MIN_CHUNK");
    if (n != 0 && ((min_keys && *min_keys) || (floor && *floor))) {
        if (plan.way == hist::Way::kFew) plan.way = hist::Way::kMerge;
        plan.chunk = hist::ChunkFor(n, floor && *floor ? strtoull(floor, nullptr, 0) : hist::ChunkFloor(n));
        plan.groups = (n + plan.chunk - 1) / plan.chunk;
        if (min_keys && *min_keys) plan.way = n >= strtoull(min_keys, nullptr, 0) ? hist::Way::kMerge : hist::Way::kSweep;
        if (plan.groups > hist::kMaxPartials) plan.way = hist::Way::kSweep;
    }
    if (plan.groups > GuardState::kMaxWorkGroups) return kXSchedErrorInvalidValue;
    *cmd = HwCommandManager::Add(std::make_shared<hist::HipHistogramCommand>(keys, n, bins, n_bins, plan, guard));
    return kXSchedSuccess;
}
