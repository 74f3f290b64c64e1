// Guarded streaming AXPY for gfx950: y = fma(alpha, x, y), fp32, in place.
//
// HBM-bound: 12 bytes of traffic per element (read x, read y, write y). The unit of
// work is a chunk of `steps` x 1024 contiguous elements, walked by one wavefront in
// steps of 4 x 128-bit accesses per lane and stream, lane-contiguous so that every
// access of a wave covers 1 KiB. Loads are non-temporal, nothing is reused; so are most
// stores (ThroughFrom()). Chunks begin on a line of y (HeadOf()).
// Because the update is in place, a chunk must be applied exactly once: the wave reads
// the preempt word before it stores anything, and commits the chunk's byte in the
// progress map after its last store.
//
// Two grids:
//   one single-wave work-group per chunk: plain launches of arrays below 2^23 elements.
//       Every chunk is in flight at once, which is what a short array wants; on long
//       arrays these short-lived waves stream at 6.2-6.3 TB/s on MI355X.
//   a few long-lived waves per CU (two, more for short arrays), each walking chunks c, c + G, c + 2G, ... with the loads
//       of three steps in flight: guarded launches, and plain launches of long arrays.
//       Same bandwidth (measured: 2 waves per CU 6.2 TB/s, 1 per CU 4.1, 4 or more per CU
//       5.3-5.8 whatever the depth), and nearly all wave slots stay free: a short kernel of
//       another queue that arrives meanwhile finishes ~10 us earlier than beside a grid of
//       262144 work-groups. A guarded launch reads the preempt word in front of every chunk:
//       after a deactivation every wave stops at its next chunk, about a microsecond away,
//       and a launch queued behind has only G work-groups to retire: the device drains in
//       6 us (p50).
//   XSCHED_HIP_AXPY_GRID=chunk keeps the first grid for everything, with the guard at
//       work-group entry: after a deactivation the device then still has to start and retire
//       every remaining work-group, empty, at ~3.3 waves per nanosecond: two launches of
//       262144 work-groups in flight drain in ~180 us.
#include "hip_hal.h"
#include "xsched/hip/hal.h"
#include "xsched/utils/env.h"

using namespace xsched::preempt;

namespace xsched::hip
{

namespace axpy
{

constexpr uint32_t kLanes = 64;
constexpr uint32_t kStepElems = 1024;                      // unit in which chunk sizes are counted

// 128-bit access unit. It is declared aligned to its elements only: a global access of 128 bits
// takes any multiple of four bytes, so slices of larger arrays run on the same kernels. Aligned
// arrays lose nothing by it (2^28 elements: 508 us, 511 with 16-byte alignment declared), arrays
// off their lines lose a few per cent where their stores are (HeadOf()).
typedef float float4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ float4 ld_nt(const float4 *p) { return __builtin_nontemporal_load(p); }
__device__ __forceinline__ void st_nt(float4 *p, float4 v) { __builtin_nontemporal_store(v, p); }

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

/// Piece u of a wave's step that begins at `first` (uniform). kThrough: the store goes through the L2 to the
/// last-level cache (device scope, sc1). A launch over a short array otherwise ends by writing back
/// what its stores left in the L2s.
template <bool kThrough>
__device__ __forceinline__ void StoreLanes(float4 *first, uint32_t lane, uint32_t u, float4 v)
{
    if constexpr (kThrough) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(first, 0, 0x7fffffff, 0x00020000);
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, (int)(lane * 16 + u * kLanes * 16), 0, 0x10);
    } else {
        st_nt(first + u * kLanes + lane, v);
    }
}

__device__ __forceinline__ float4 fma4(float a, float4 x, float4 y)
{
    float4 r;
    r.x = __builtin_fmaf(a, x.x, y.x);
    r.y = __builtin_fmaf(a, x.y, y.y);
    r.z = __builtin_fmaf(a, x.z, y.z);
    r.w = __builtin_fmaf(a, x.w, y.w);
    return r;
}

// n4: number of whole float4 in the arrays; tail: the 0..3 trailing scalars, done by
// the last work-group; head: elements in front of x_first and y_first, done with chunk 0 (HeadOf()).
// kVecPerStep float4 per lane and stream are requested before anything is stored:
// 4 -> steps of 1024 elements, 8 -> steps of 2048 elements.
template <bool kGuard, uint32_t kVecPerStep, bool kThrough>
__global__ __launch_bounds__(64)
void AxpyVec4Kernel(float alpha, const float *x_first, float *y_first,
                    uint64_t n4, uint32_t tail, uint32_t head, uint32_t steps, XGuardArgs g)
{
    const float4 *const x = (const float4 *)x_first;
    float4 *const y = (float4 *)y_first;
    constexpr uint32_t kStepVecs = kLanes * kVecPerStep;
    const uint32_t wg = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const uint64_t wg_base = (uint64_t)wg * steps * kStepVecs;
    XGuardWave guard(g, wg);

    const bool full = wg_base + (uint64_t)steps * kStepVecs <= n4;
    // The guard comes before the loads: a flushed work-group then costs no memory
    // traffic at all, which keeps the drain after a deactivation short; with 8 waves per
    // SIMD the extra round trip does not show in the bandwidth (measured).
    if (kGuard) {
        if (!guard.Enter()) return;
    }
    if (wg == 0 && lane < head) {
        const float *const xs = x_first - head;
        float *const ys = y_first - head;
        ys[lane] = __builtin_fmaf(alpha, xs[lane], ys[lane]);
    }
    if (full) {
        for (uint32_t s = 0; s < steps; ++s) {
            const uint64_t base = wg_base + (uint64_t)s * kStepVecs + lane;
            float4 xv[kVecPerStep], yv[kVecPerStep];
#pragma unroll
            for (uint32_t u = 0; u < kVecPerStep; ++u) {
                xv[u] = ld_nt(&x[base + u * kLanes]);
                yv[u] = ld_nt(&y[base + u * kLanes]);
            }
#pragma unroll
            for (uint32_t u = 0; u < kVecPerStep; ++u) {
                StoreLanes<kThrough>(y + wg_base + (uint64_t)s * kStepVecs, lane, u, fma4(alpha, xv[u], yv[u]));
            }
        }
    } else {
        const uint64_t end = wg_base + (uint64_t)steps * kStepVecs;
        for (uint64_t i = wg_base + lane; i < end && i < n4; i += kLanes) {
            st_nt(&y[i], fma4(alpha, ld_nt(&x[i]), ld_nt(&y[i])));
        }
        if (wg == gridDim.x - 1 && lane < tail) {
            const float *xs = (const float *)(x + n4);
            float *ys = (float *)(y + n4);
            ys[lane] = __builtin_fmaf(alpha, xs[lane], ys[lane]);
        }
    }
    if (kGuard) guard.Commit();
}

// Guarded launches: grid-stride over chunks, see the head of this file. `n_chunks`
// chunks of `steps` x 1024 elements; the progress map has one byte per chunk.
// A wave walks its chunks c, c + G, c + 2G, ... step by step and keeps the loads of
// kDepth steps in flight: step j is stored while steps j+1 .. j+kDepth-1 are on their
// way and step j+kDepth is requested right behind the stores. The preempt word is read
// in front of the first store of every chunk; a chunk that has begun is finished and
// committed, so it is applied exactly once.
// kThrough: the chunks from `through` on are stored through the L2, which holds nothing to be
// written back of them when the kernel ends (ThroughFrom()).
template <uint32_t kDepth, bool kGuard, bool kThrough>
__global__ __launch_bounds__(64)
void AxpyPersistentKernel(float alpha, const float *x_first, float *y_first, uint64_t n4, uint32_t tail,
                          uint32_t head, uint32_t steps, uint32_t n_chunks, uint32_t through, XGuardArgs g)
{
    const float4 *const x = (const float4 *)x_first;
    float4 *const y = (float4 *)y_first;
    constexpr uint32_t kVecPerStep = 4;
    constexpr uint32_t kStepVecs = kLanes * kVecPerStep;
    const uint32_t lane = threadIdx.x;
    const uint32_t stride = gridDim.x;
    const uint32_t *flag = kGuard ? xguard_flag_copy(g, blockIdx.x) : nullptr;

    // Ring slot d holds step ring_s[d] of chunk ring_c[d]; the slots follow each other in
    // the wave's sequence of steps.
    uint32_t ring_c[kDepth], ring_s[kDepth];
    float4 xv[kDepth][kVecPerStep], yv[kDepth][kVecPerStep];
    {
        uint32_t c = blockIdx.x, st = 0;
#pragma unroll
        for (uint32_t d = 0; d < kDepth; ++d) {
            ring_c[d] = c;
            ring_s[d] = st;
            if (++st == steps) { st = 0; c += stride; }
        }
    }
#pragma unroll
    for (uint32_t d = 0; d < kDepth; ++d) {
        const uint32_t c = ring_c[d];
        if (c < n_chunks && ((uint64_t)c + 1) * steps * kStepVecs <= n4) {
            const uint64_t base = ((uint64_t)c * steps + ring_s[d]) * kStepVecs + lane;
#pragma unroll
            for (uint32_t u = 0; u < kVecPerStep; ++u) {
                xv[d][u] = ld_nt(&x[base + u * kLanes]);
                yv[d][u] = ld_nt(&y[base + u * kLanes]);
            }
        }
    }

    // An earlier launch of this epoch was flushed: this one must not run ahead of its replay. (Looked at behind
    // the first loads, which have no side effect: a scalar load, so nobody waits for them.)
    if (kGuard && xguard_epoch_flushed(g)) return;

    bool skip = false;   // the chunk whose steps are passing by was committed before the flush
    while (true) {
        // no unroll pragma here: the constant trip count is unrolled anyway, and with the
        // pragma the compiler warns about a copy of the loop that it drops afterwards
        for (uint32_t d = 0; d < kDepth; ++d) {
            const uint32_t c = ring_c[d];
            const uint32_t st = ring_s[d];
            if (c >= n_chunks) return;   // the sequence only grows: every later step is beyond, too
            const bool full = ((uint64_t)c + 1) * steps * kStepVecs <= n4;
            if (st == 0) {
                // The scalar read of the preempt word waits for itself only: the vector loads
                // stay in flight across it. A flushed wave drops what it has loaded.
                if (kGuard) {
                    const XGuardVerdict v = xguard_recheck_verdict(xguard_read_flag(flag), g.epoch);
                    if (v.note_flush && lane == 0) xguard_note_flush(g);
                    if (!v.run) return;
                    skip = g.resume && g.done && xguard_committed(g, c);
                }
                if (!skip && c == 0 && lane < head) {
                    const float *const xs = x_first - head;
                    float *const ys = y_first - head;
                    ys[lane] = __builtin_fmaf(alpha, xs[lane], ys[lane]);
                }
                if (!skip && !full) {
                    // the last chunk of an array that does not fill it, and the 0..3 scalars behind
                    const uint64_t chunk_base = (uint64_t)c * steps * kStepVecs;
                    const uint64_t end = chunk_base + (uint64_t)steps * kStepVecs;
                    for (uint64_t i = chunk_base + lane; i < end && i < n4; i += kLanes) {
                        st_nt(&y[i], fma4(alpha, ld_nt(&x[i]), ld_nt(&y[i])));
                    }
                    if (c == n_chunks - 1 && lane < tail) {
                        const float *xs = (const float *)(x + n4);
                        float *ys = (float *)(y + n4);
                        ys[lane] = __builtin_fmaf(alpha, xs[lane], ys[lane]);
                    }
                    if (kGuard && g.done && lane == 0) xguard_commit(g, c);
                }
            }
            if (full && !skip) {
                float4 *const first = y + ((uint64_t)c * steps + st) * kStepVecs;
                if (kThrough && c >= through) {
#pragma unroll
                    for (uint32_t u = 0; u < kVecPerStep; ++u) StoreLanes<true>(first, lane, u, fma4(alpha, xv[d][u], yv[d][u]));
                } else {
#pragma unroll
                    for (uint32_t u = 0; u < kVecPerStep; ++u) StoreLanes<false>(first, lane, u, fma4(alpha, xv[d][u], yv[d][u]));
                }
                if (kGuard && st == steps - 1 && g.done && lane == 0) xguard_commit(g, c);
            }
            // this slot's next step: kDepth steps further on in the sequence
            uint32_t nc = c, ns = st + kDepth;
            while (ns >= steps) { ns -= steps; nc += stride; }
            ring_c[d] = nc;
            ring_s[d] = ns;
            if (nc < n_chunks && ((uint64_t)nc + 1) * steps * kStepVecs <= n4) {
                const uint64_t nb = ((uint64_t)nc * steps + ns) * kStepVecs + lane;
#pragma unroll
                for (uint32_t u = 0; u < kVecPerStep; ++u) {
                    xv[d][u] = ld_nt(&x[nb + u * kLanes]);
                    yv[d][u] = ld_nt(&y[nb + u * kLanes]);
                }
            }
        }
    }
}

class HipAxpyCommand final : public HipGuardedCommand
{
public:
    /// steps: chunk size per work-group in units of 1024 elements.
    /// head: HeadOf(), which the chunks do not count.
    HipAxpyCommand(float alpha, const float *x, float *y, size_t n, uint32_t head, uint32_t steps, uint32_t n_wg,
                   int guard_mode, bool chunk_grid)
        : HipGuardedCommand(n_wg, guard_mode), alpha_(alpha), x_(x), y_(y), n_(n), head_(head), steps_(steps)
        , chunk_grid_(chunk_grid) {}

    /// Elements of y in front of its first 128-byte line. Chunks begin behind them, so that a wave's stores cover whole lines:
    /// of an array off its lines each store of 1 KiB began and ended inside a line, which two waves then
    /// wrote in pieces. us per command in a stream of them from an odd offset, without and with it (and with the stores of ThroughFrom()), on one pair of arrays and on 800 MB
    /// in turn: level 1 2^20 elements 4.6 / 4.2 and 5.7 / 5.3, 3 x 2^20 7.0 / 5.6 and 9.2 / 8.5, 6 x 2^20 13.0 / 12.3 and 15.2 / 14.5, 2^23 17.2 / 16.5
    /// and 19.1 / 18.6, 2^24 33.2 / 29.7 and 34.8 / 31.3, 2^25 67.9 / 65.9 and 68.4 / 66.2; level 2 3 x 2^20 7.6 / 7.5 and 9.4 / 9.2, 2^24 33.6 / 31.0 and 35.2 / 32.6.
    /// (All of 2^24 through the L2 without it: 31.4 and 39.6.)
    static uint32_t HeadOf(const float *y, size_t n)
    {
        const uint32_t off = (uint32_t)((uintptr_t)y & 127);
        if (off == 0 || off % 4 != 0) return 0;
        const uint32_t head = (128 - off) / 4;
        return n < head ? (uint32_t)n : head;
    }

    static bool WavePerChunk(bool guarded, uint32_t n_wg, bool chunk_grid) { return chunk_grid || (!guarded && n_wg < kLongChunks); }

    /// First chunk whose stores go through the L2 (n_wg: none). On one wave per chunk all of them, of arrays of up to kThroughTo elements, from a size on that depends on
    /// whether they begin on a line. us per command in a stream of them, on one pair of arrays / on pairs of 800 MB in turn (nothing is in
    /// the last-level cache then), and of a pass alone, on one pair / behind a fill of 640 MB, non-temporal stores -> these: on a line 2^20 elements 4.20 / 4.50, 13.0 / 16.5 ->
    /// 4.09 / 4.53, 13.3 / 15.6 (runs differ by 0.1 to 0.3), 5 x 2^18 4.31 / 4.72, 13.6 / 16.5 -> 4.33 / 4.92, 13.6 / 16.1, 2^21 4.75 / 6.30, 14.0 / 18.1 -> 4.76 / 6.18,
    /// 14.7 / 17.3, 5 x 2^19 5.97 / 7.67, 16.1 / 19.7 -> 5.25 / 7.43, 16.3 / 18.9, 2^22 8.40 / 10.3, 18.3 / 22.3 -> 6.57 / 10.1, 18.2 / 21.7; off a line 2^20
    /// 4.60 / 5.39, 13.4 / 17.4 -> 4.71 / 5.19, 13.6 / 16.7, 5 x 2^18 5.21 / 5.88, 15.7 / 19.7 -> 4.81 / 5.72, 15.8 / 18.6, 2^21 5.83 / 7.21, 15.9 / 19.3 ->
    /// 4.86 / 6.84, 15.6 / 18.5. Traced, a launch of 2^16 elements takes 2.5 us with these and 2.1 without.
    /// Above, level 1 6 x 2^20 10.9 / 13.8 -> 11.5 / 13.9.
    /// On long-lived waves, eight per compute unit, for more than 32768 and up to 65536 elements per unit (2^23 and 2^24 on 256): the last three
    /// quarters of the chunks. Non-temporal -> all of them -> these, the same four figures: level 1 2^23 + 1024 elements 16.0 / 17.8, 27.5 / 28.9 -> 14.0 / 18.4, 23.7 / 28.9 ->
    /// 15.1 / 17.9, 24.3 / 29.3; 12 x 2^20 24.3 / 25.8, 35.4 / 37.2 -> 21.0 / 26.6, 30.0 / 37.4 -> 22.1 / 24.2, 31.0 / 37.4; 2^24 31.3 / 33.1, 42.4 / 45.0 ->
    /// 28.8 / 34.2, 38.9 / 46.1 -> 29.3 / 30.9, 38.3 / 45.4; level 2 2^23 + 1024 16.0 / 18.4, 28.4 / 29.8 -> 14.6 / 18.7, 24.7 / 29.8 -> 15.0 / 18.3, 25.6 / 29.8;
    /// 2^24 31.4 / 33.5, 43.5 / 44.9 -> 29.1 / 34.6, 39.4 / 46.2 -> 30.7 / 32.2, 39.4 / 46.4. So arrays that are not in the last-level cache, which lost 2 % to 3 % with
    /// all chunks through, gain up to 7 % where they follow each other, and single passes over them lose up to 1.5 us (runs differ by 1); with a half or five
    /// eighths of the chunks passes on one pair gain up to 2 us less. 5000 elements longer it is non-temporal stores and two waves per unit: 33.5 / 35.0, 44.9 / 46.3.
    static uint32_t ThroughFrom(size_t n, uint32_t head, uint32_t n_wg, bool wave_per_chunk, uint32_t units)
    {
        if (wave_per_chunk) return n > (head != 0 ? kThroughOffLines : kThroughOnLines) && n <= kThroughTo ? 0 : n_wg;
        if (n <= (uint64_t)32 * kStepElems * units || n > (uint64_t)64 * kStepElems * units) return n_wg;
        return n_wg / 4;
    }

    /// Long-lived waves of a launch over n_wg chunks: two per compute unit for long arrays, more
    /// while each has only a few chunks, where what counts is how many requests are out at once
    /// (us per command at level 2 in a stream of them, on one pair of arrays / on 800 MB of them, at 2, 4, 8, 12 waves per CU and with non-temporal
    /// stores: 2^21 elements 5.7 / 7.1, 5.4 / 6.7, 5.2 / 6.3, 5.2 / 6.3; 2^22 10.2 / 11.6, 9.1 / 10.7, 8.4 / 10.3, 8.2 / 10.0; 6 x 2^20 14.4 / 15.8, 13.1 / 14.8,
    /// 12.9 / 14.7, 12.6 / 14.6; 2^23 18.4 / 19.7, 16.9 / 18.6, 16.9 / 18.9, 16.3 / 18.1; 2^25 69.3, 67.4, 67.3, 69.7; 2^28 513, 554, 558, 569). `through`: with
    /// stores through the L2, which the loads of a guarded launch's wave wait for, 2^24 takes 32.1 with four and 29.1 with eight.
    static uint32_t WavesFor(uint32_t n_wg, bool through, uint32_t units)
    {
        return (through || n_wg <= 16 * units ? 8 : n_wg <= 64 * units ? 4 : 2) * units;
    }

protected:
    virtual hipError_t LaunchKernel(hipStream_t stream, bool guarded, const XGuardArgs &g) override
    {
        if (n_ == 0) return hipSuccess;
        const hipEvent_t stop = TakeStopEvent();
        const uint32_t through = ThroughFrom(n_, head_, n_wg_, WavePerChunk(guarded, n_wg_, chunk_grid_), ComputeUnits());
        if (through < n_wg_) Launch<true>(guarded, stop, stream, through, g);
        else Launch<false>(guarded, stop, stream, through, g);
        return hipGetLastError();
    }

private:
    template <bool kThrough>
    void Launch(bool guarded, hipEvent_t stop, hipStream_t stream, uint32_t through, const XGuardArgs &g)
    {
        const dim3 grid(n_wg_), block(kLanes);
        const uint32_t waves = PersistentWaves(n_wg_, kThrough);
        const float *const x = x_ + head_;
        float *const y = y_ + head_;
        const uint64_t n4 = (n_ - head_) / 4;
        const uint32_t tail = (uint32_t)((n_ - head_) % 4);
        if (guarded && !chunk_grid_) {
            const dim3 pgrid(n_wg_ < waves ? n_wg_ : waves);
            LaunchWithStop(stop, (AxpyPersistentKernel<3, true, kThrough>), pgrid, block, stream, alpha_, x, y, n4, tail, head_, steps_, n_wg_, through, g);
        } else if (!guarded && !chunk_grid_ && n_wg_ >= kLongChunks) {
            // A long array: the same few long-lived waves stream it as fast as one wave per
            // chunk does and leave nearly all wave slots to whatever else runs on the device.
            LaunchWithStop(stop, (AxpyPersistentKernel<3, false, kThrough>), dim3(waves), block, stream, alpha_, x, y, n4, tail, head_, steps_, n_wg_, through, g);
        } else {
            // An even chunk is walked in steps of 2048 elements (8 accesses in flight
            // per lane and stream), an odd one in steps of 1024.
            const bool wide = (steps_ % 2) == 0;
            const uint32_t steps = wide ? steps_ / 2 : steps_;
            if (guarded && wide)       LaunchWithStop(stop, (AxpyVec4Kernel<true, 8, kThrough>), grid, block, stream, alpha_, x, y, n4, tail, head_, steps, g);
            else if (guarded)          LaunchWithStop(stop, (AxpyVec4Kernel<true, 4, kThrough>), grid, block, stream, alpha_, x, y, n4, tail, head_, steps, g);
            else if (wide)             LaunchWithStop(stop, (AxpyVec4Kernel<false, 8, kThrough>), grid, block, stream, alpha_, x, y, n4, tail, head_, steps, g);
            else                       LaunchWithStop(stop, (AxpyVec4Kernel<false, 4, kThrough>), grid, block, stream, alpha_, x, y, n4, tail, head_, steps, g);
        }
    }

    static uint32_t ComputeUnits()
    {
        static const uint32_t cus = []() {
            int dev = 0, n = 256;
            if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
            return (uint32_t)(n > 0 ? n : 256);
        }();
        return cus;
    }

    static uint32_t PersistentWaves(uint32_t n_wg, bool through)
    {
        static const int64_t asked = []() {
            int64_t per_cu = 0;
            GetEnvInt64("XSCHED_HIP_AXPY_WAVES_PER_CU", per_cu);
            return per_cu < 0 ? (int64_t)1 : per_cu > 64 ? (int64_t)64 : per_cu;
        }();
        return asked > 0 ? (uint32_t)asked * ComputeUnits() : WavesFor(n_wg, through, ComputeUnits());
    }

    static constexpr uint64_t kThroughOffLines = (uint64_t)1 << 20, kThroughOnLines = (uint64_t)1 << 21, kThroughTo = (uint64_t)1 << 22;
    static constexpr uint32_t kLongChunks = 8192;   // from here on a plain launch uses long-lived waves

    const float alpha_;
    const float *x_;
    float *y_;
    const size_t n_;
    const uint32_t head_;
    const uint32_t steps_;
    const bool chunk_grid_;   // guarded launches keep the one-wave-per-chunk grid
};

} // namespace axpy

using namespace axpy;

/// Steps (of 1024 elements) per work-group: small enough that the device drains in
/// tens of microseconds after a flush, large enough that the grid fits the progress
/// map.
uint32_t AxpyStepsFor(size_t n)
{
    int64_t dflt = 1;
    GetEnvInt64("XSCHED_HIP_AXPY_STEPS", dflt);
    uint64_t steps = (uint64_t)(dflt < 1 ? 1 : dflt);
    while (((uint64_t)n + steps * kStepElems - 1) / (steps * kStepElems) > GuardState::kMaxWorkGroups) steps *= 2;
    return (uint32_t)steps;
}

} // namespace xsched::hip

using namespace xsched::hip;

EXPORT_C_FUNC XResult HipAxpyCommandCreate(HwCommandHandle *cmd, float alpha, const void *x, void *y,
                                           size_t n, int guard)
{
    if (cmd == nullptr || (n != 0 && (x == nullptr || y == nullptr)) || guard < 0 || guard > 3) {
        return kXSchedErrorInvalidValue;
    }
    const uint32_t head = axpy::HipAxpyCommand::HeadOf((const float *)y, n);
    const uint32_t steps = AxpyStepsFor(n - head);
    const uint64_t per_wg = (uint64_t)steps * 1024;
    const uint32_t n_wg = n == head ? 1 : (uint32_t)((n - head + per_wg - 1) / per_wg);
    *cmd = HwCommandManager::Add(std::make_shared<axpy::HipAxpyCommand>(
        alpha, (const float *)x, (float *)y, n, head, steps, n_wg, guard, GetEnv("XSCHED_HIP_AXPY_GRID") == "chunk"));
    return kXSchedSuccess;
}

EXPORT_C_FUNC XResult HipAxpyPlanOf(const void *y, size_t n, int guarded, uint32_t compute_units, uint32_t *out)
{
    if (out == nullptr || n == 0 || compute_units == 0) return kXSchedErrorInvalidValue;
    using Command = axpy::HipAxpyCommand;
    const uint32_t head = Command::HeadOf((const float *)y, n), steps = AxpyStepsFor(n - head);
    const uint64_t per_wg = (uint64_t)steps * 1024;
    const uint32_t chunks = n == head ? 1 : (uint32_t)((n - head + per_wg - 1) / per_wg);
    const bool wave_per_chunk = Command::WavePerChunk(guarded != 0, chunks, GetEnv("XSCHED_HIP_AXPY_GRID") == "chunk");
    out[0] = chunks;
    out[2] = Command::ThroughFrom(n, head, chunks, wave_per_chunk, compute_units);
    out[1] = wave_per_chunk ? 0 : Command::WavesFor(chunks, out[2] < chunks, compute_units);
    return kXSchedSuccess;
}
