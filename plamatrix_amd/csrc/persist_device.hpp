// Device pieces of the persistent solves: the words that cross workgroups, the
// bounded waits, and the decision and reduction phases of an iteration.
#pragma once

#include "persist_history.hpp"
#include "spmv_kernels.hpp"

namespace pm
{

using word = unsigned long long;

constexpr int kPersistThreads = 1024;
constexpr int kPersistWaves = kPersistThreads / kWave;
constexpr int kPersistGroups = kPersistThreads / kBlock;  // per-kernel workgroups one workgroup stands for
constexpr int kPersistBlocks = kSolverGrid / kPersistGroups;
constexpr int kRedEntries = kSolverGrid - kBlock;
constexpr int kDecWords = 16;        // one 128-byte line per workgroup
constexpr int kWaitSeconds = 4;
constexpr int64_t kSegment = 8192;   // iterations per launch
constexpr size_t kPersistLds = 160 * 1024 - 2048;  // LDS of a CU less the static part

struct PersistControl
{
    unsigned abort;
    unsigned finished;
    unsigned pad[62];
    word part[2][kCgValues][2][kSolverGrid];  // parity, value, half, per-kernel workgroup
    word dec[kPersistBlocks][kDecWords];
};

__device__ __forceinline__ word load_word(const word* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void store_word(word* p, unsigned v, unsigned tag)
{
    __hip_atomic_store(p, (static_cast<word>(tag) << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Word i of an exchange array (fewer than 2^29 words: a 32-bit byte offset from
// a uniform base).
__device__ __forceinline__ word* word_at(word* b, unsigned i)
{
    return reinterpret_cast<word*>(reinterpret_cast<char*>(b) + i * 8u);
}
__device__ __forceinline__ const word* word_at(const word* b, unsigned i)
{
    return reinterpret_cast<const word*>(reinterpret_cast<const char*>(b) + i * 8u);
}
__device__ __forceinline__ bool word_ready(word v, unsigned tag) { return static_cast<unsigned>(v >> 32) == tag; }

// A value of the exchange: one word for FP32, two for FP64 (half planes).
template <typename S>
struct Exchange;
template <>
struct Exchange<float>
{
    static constexpr int kWords = 1;
    __device__ static __forceinline__ void put(word* b, int, unsigned i, float v, unsigned tag)
    {
        store_word(word_at(b, i), __float_as_uint(v), tag);
    }
    __device__ static __forceinline__ void issue(const word* b, int, unsigned i, word (&w)[1])
    {
        w[0] = load_word(word_at(b, i));
    }
    __device__ static __forceinline__ float value(const word (&w)[1]) { return __uint_as_float(static_cast<unsigned>(w[0])); }
};
template <>
struct Exchange<double>
{
    static constexpr int kWords = 2;
    __device__ static __forceinline__ void put(word* b, int plane, unsigned i, double v, unsigned tag)
    {
        const word bits = static_cast<word>(__double_as_longlong(v));
        store_word(word_at(b, i), static_cast<unsigned>(bits), tag);
        store_word(word_at(b + plane, i), static_cast<unsigned>(bits >> 32), tag);
    }
    __device__ static __forceinline__ void issue(const word* b, int plane, unsigned i, word (&w)[2])
    {
        w[0] = load_word(word_at(b, i));
        w[1] = load_word(word_at(b + plane, i));
    }
    __device__ static __forceinline__ double value(const word (&w)[2])
    {
        return __longlong_as_double(static_cast<long long>((w[1] << 32) | (w[0] & 0xffffffffull)));
    }
};
template <typename S>
__device__ __forceinline__ bool ready(const word (&w)[Exchange<S>::kWords], unsigned tag)
{
    bool ok = word_ready(w[0], tag);
    if constexpr (Exchange<S>::kWords == 2) ok = ok && word_ready(w[1], tag);
    return ok;
}

// The workgroup of the per-kernel iteration that owns logical block lb (the
// inverse of xcd_logical_block).
__device__ __forceinline__ int physical_block(int lb, int nb)
{
    const int q = nb / kXcds, r = nb % kXcds;
    const int head = r * (q + 1);
    const int xcd = lb < head ? lb / (q + 1) : r + (lb - head) / (q > 0 ? q : 1);
    const int idx = lb < head ? lb % (q + 1) : (lb - head) % (q > 0 ? q : 1);
    return idx * kXcds + xcd;
}

// Waits for words that other workgroups write: `poll` loads them and says
// whether all carry their tag.  The whole wavefront polls together.  `abort`: the
// launch's notice to give up.
template <typename Poll>
__device__ __forceinline__ bool wait_for(unsigned* abort, Poll poll)
{
    unsigned polls = 0;
    long long start = 0;
    while (!__all(poll()))
    {
        // the bound of the wait: every 256 polls look at the clock (100 MHz)
        // and at another workgroup's notice that it gave up
        if ((++polls & 255u) != 0u) continue;
        const long long now = wall_clock64();
        if (start == 0) start = now;
        if (__hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u ||
            now - start > kWaitSeconds * 100000000ll)
        {
            __hip_atomic_store(abort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return false;
        }
    }
    return true;
}

// Whether another workgroup already gave up: a workgroup that starts late leaves at its
// first decision (no exit of its own before: it costs the solve kernels registers).
__device__ __forceinline__ int given_up(const unsigned* abort)
{
    return __hip_atomic_load(abort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u ? 1 : 0;
}

// The workgroup-shared part of a persistent solve.
template <typename S>
struct PersistShared
{
    double part[kCgValues][kPersistWaves];   // partial sums of the wavefronts
    double sum[kCgValues][kBlock / kWave];   // the decision's reduction
    S alpha, beta;
    int code, fail;
    PersistHistory hs;
};

// Where a workgroup stands in the launch.
struct PersistWhere
{
    PersistControl* ctl;
    double* region;  // partials of iteration t0 - 1
    int bid, blocks, g;  // workgroup, its piece
    int count, leaders;  // per-kernel workgroups, workgroups that decide
    int t0, chunk, grow;
};

// The decision at the head of iteration t, from the partials of t - 1: leading
// workgroups reduce and decide, the rest receive alpha, beta and the code.
// `red`: LDS for NV * kRedEntries doubles where there are more than kBlock
// partials.  Ends with a workgroup barrier; false: give up.
template <typename S, int NV>
__device__ __forceinline__ bool persist_decide(PersistShared<S>& sh, const PersistWhere& at, int t, unsigned tag,
                                               double* red)
{
    using X = Exchange<S>;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    if (at.bid < at.leaders)
    {
        bool fine = true;
        auto entry = [&](int e, double (&out)[NV]) {
            if (t == at.t0)
            {
#pragma unroll
                for (int v = 0; v < NV; ++v) out[v] = at.region[(NV == 3 && v > 0 ? v + 1 : v) * kMaxPartials + e];
                return;
            }
            word hw[NV][2];
            const word* from = &at.ctl->part[(t - 1) & 1][0][0][e];
            fine = wait_for(&at.ctl->abort, [&] {
                bool ok = true;
#pragma unroll
                for (int v = 0; v < NV; ++v)
                {
                    hw[v][0] = load_word(from + (2 * v) * kSolverGrid);
                    hw[v][1] = load_word(from + (2 * v + 1) * kSolverGrid);
                }
#pragma unroll
                for (int v = 0; v < NV; ++v)
                    ok = ok && word_ready(hw[v][0], tag - 1u) && word_ready(hw[v][1], tag - 1u);
                return ok;
            });
#pragma unroll
            for (int v = 0; v < NV; ++v) out[v] = Exchange<double>::value(hw[v]);
        };
        double acc[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[v] = 0.0;
        if (at.count <= kBlock)
        {
            if (tid < at.count)
            {
                double e[NV];
                entry(tid, e);
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[v] += e[v];
            }
        }
        else
        {
            double e[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v) e[v] = 0.0;
            if (tid < at.count) entry(tid, e);
            if (tid >= kBlock)
            {
#pragma unroll
                for (int v = 0; v < NV; ++v) red[v * kRedEntries + tid - kBlock] = e[v];
            }
            __syncthreads();
            if (tid < kBlock)
            {
#pragma unroll
                for (int v = 0; v < NV; ++v)
                {
                    acc[v] += e[v];
#pragma unroll
                    for (int j = 0; j < kRedEntries / kBlock; ++j) acc[v] += red[v * kRedEntries + tid + j * kBlock];
                }
            }
        }
        if (tid < kBlock)
        {
            const double sum = wave_sum4(acc[0], acc[1], acc[2], acc[NV - 1]);
            if (lane % 16 == 0) sh.sum[lane / 16][wave] = sum;
        }
        if (!fine) sh.fail = 1;
        __syncthreads();
        if (tid == 0)
        {
            double tot[NV];
#pragma unroll
            for (int v = 0; v < NV; ++v)
            {
                double q = 0.0;
#pragma unroll
                for (int z = 0; z < kBlock / kWave; ++z) q += sh.sum[v][z];
                tot[v] = q;
            }
            sh.code = sh.hs.template decide<S>(t, tot[0], tot[NV == 4 ? 1 : 0], tot[NV - 2], tot[NV - 1], at.chunk,
                                               at.grow != 0, sh.alpha, sh.beta);
        }
        __syncthreads();
        // the workgroups this leader answers to: bid + leaders, ...
        const int who = at.bid + (tid + 1) * at.leaders;
        if (who < at.blocks && sh.fail == 0)
        {
            word* line = at.ctl->dec[who];
            X::put(line, kDecWords / 2, 0, sh.alpha, tag);
            X::put(line, kDecWords / 2, 1, sh.beta, tag);
            store_word(line + 2, static_cast<unsigned>(sh.code), tag);
        }
    }
    else
    {
        if (wave == 0)
        {
            // alpha, beta, code by lanes 0, 1, 2 (the other lanes repeat 2)
            const word* line = at.ctl->dec[at.bid] + (lane < 2 ? lane : 2);
            word hw[X::kWords];
            const bool fine = wait_for(&at.ctl->abort, [&] {
                hw[0] = load_word(line);
                bool ok = word_ready(hw[0], tag);
                if constexpr (X::kWords == 2)
                {
                    hw[1] = load_word(line + (lane < 2 ? kDecWords / 2 : 0));
                    ok = ok && word_ready(hw[1], tag);
                }
                return ok;
            });
            if (!fine) sh.fail = 1;
            if (lane == 0) sh.alpha = X::value(hw);
            else if (lane == 1) sh.beta = X::value(hw);
            else if (lane == 2) sh.code = static_cast<int>(hw[0]);
        }
        __syncthreads();
    }
    return sh.fail == 0;
}

// The lanes' partial sums of iteration t, summed per per-kernel workgroup and
// published.  Holds a workgroup barrier; false: give up.
template <typename S, int NV>
__device__ __forceinline__ bool persist_partials(PersistShared<S>& sh, const PersistWhere& at, int t, unsigned tag,
                                                 const double (&part)[kCgValues])
{
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const double sum = wave_sum4(part[0], part[1], part[2], part[NV - 1]);
    if (lane % 16 == 0) sh.part[lane / 16][wave] = sum;
    __syncthreads();
    if (sh.fail != 0) return false;
    if (tid < NV * kPersistGroups)
    {
        const int v = tid / kPersistGroups, q = tid % kPersistGroups;
        const int lb = at.g * kPersistGroups + q;
        if (lb < at.count)
        {
            double group = 0.0;
#pragma unroll
            for (int z = 0; z < kWavesPerBlock; ++z) group += sh.part[v][q * kWavesPerBlock + z];
            const int vb = physical_block(lb, at.count);
            Exchange<double>::put(&at.ctl->part[t & 1][v][0][vb], kSolverGrid, 0, group, tag);
        }
    }
    return true;
}

// After a hand-over: the workgroup's last partials where the three-kernel form
// reads them.  t0 and the hand-over iteration are even, so they are of an odd
// iteration, region 1.
template <int NV>
__device__ __forceinline__ void persist_leave_partials(const PersistWhere& at)
{
    const int tid = threadIdx.x;
    if (tid >= kPersistGroups || at.g * kPersistGroups + tid >= at.count) return;
    const int vb = physical_block(at.g * kPersistGroups + tid, at.count);
    double vals[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v)
    {
        word hw[2] = {load_word(&at.ctl->part[1][v][0][vb]), load_word(&at.ctl->part[1][v][1][vb])};
        vals[v] = Exchange<double>::value(hw);
    }
    at.region[vb] = vals[0];
    at.region[kMaxPartials + vb] = vals[NV == 4 ? 1 : 0];
    at.region[2 * kMaxPartials + vb] = vals[NV - 2];
    at.region[3 * kMaxPartials + vb] = vals[NV - 1];
}

// The last step of a workgroup that reached the end of its launch.
template <typename S>
__device__ __forceinline__ void persist_end(PersistShared<S>& sh, const PersistWhere& at, SolverState* st, int code)
{
    if (at.bid == 0 && threadIdx.x == 0) sh.hs.record(st, code);
    __syncthreads();
    if (threadIdx.x == 0) __hip_atomic_fetch_add(&at.ctl->finished, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

} // namespace pm
