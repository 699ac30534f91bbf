// Shared helpers of the gfx950 library: status plumbing for the C ABI,
// deterministic wavefront/workgroup reductions, XCD-aware block numbering and
// the grow-only device buffers the workspaces own.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

#include "plamatrix_amd.h"

namespace pm
{

constexpr int kWave = 64;       // CDNA wavefront width
constexpr int kBlock = 256;     // threads per workgroup for streaming kernels
constexpr int kXcds = 8;        // MI355X: 8 XCDs, blocks dispatched round-robin
constexpr int kMaxPartials = 2048;  // upper bound on workgroups that publish partial sums

// ---- host-side status ----------------------------------------------------
void set_error(int code, const std::string& message);
int fail(int code, const char* fmt, ...);
int check_hip(hipError_t err, const char* what, const char* file, int line);

#define PM_HIP(call)                                                                     \
    do                                                                                   \
    {                                                                                    \
        hipError_t pm_err_ = (call);                                                     \
        if (pm_err_ != hipSuccess) return ::pm::check_hip(pm_err_, #call, __FILE__, __LINE__); \
    } while (0)

#define PM_TRY(expr)                         \
    do                                       \
    {                                        \
        int pm_status_ = (expr);             \
        if (pm_status_ != PM_OK) return pm_status_; \
    } while (0)

// ---- XCD-aware block numbering -------------------------------------------
// The dispatcher hands workgroup b to XCD (b % 8).  Renumbering so that each
// XCD walks one contiguous range of logical blocks keeps neighbouring rows (and
// the x entries they gather) in the same L2.
__device__ __forceinline__ int64_t xcd_logical_block(int64_t b, int64_t nb)
{
    const int64_t q = nb / kXcds;
    const int64_t r = nb % kXcds;
    const int64_t xcd = b % kXcds;
    const int64_t idx = b / kXcds;
    return xcd * q + (xcd < r ? xcd : r) + idx;
}

// LDS hand-off between lanes of one wavefront.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---- deterministic reductions ---------------------------------------------
// One step of a butterfly sum: v plus the v of lane ^ OFF, the steps taken from
// 32 down to 1.  The exchanges stay inside the vector unit (half and row swaps,
// rotations of a 16-lane row, quad permutations) instead of passing through the
// LDS crossbar; once the larger offsets are summed v repeats every 2 * OFF
// lanes, so a rotation by OFF reaches the partner's value.
template <int OFF>
__device__ __forceinline__ void butterfly_pair(unsigned v, unsigned& a, unsigned& b)
{
    if constexpr (OFF == 32 || OFF == 16)
    {
        const auto both = OFF == 32 ? __builtin_amdgcn_permlane32_swap(v, v, false, false)
                                    : __builtin_amdgcn_permlane16_swap(v, v, false, false);
        a = both[0];
        b = both[1];
    }
    else
    {
        constexpr int ctrl = OFF == 8 ? 0x128 : OFF == 4 ? 0x124 : OFF == 2 ? 0x4e : 0xb1;
        a = v;
        b = static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), ctrl, 0xf, 0xf, false));
    }
}

template <int OFF, typename T>
__device__ __forceinline__ T butterfly_add(T v)
{
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "butterfly word");
    if constexpr (sizeof(T) == 4)
    {
        unsigned a, b;
        butterfly_pair<OFF>(__builtin_bit_cast(unsigned, v), a, b);
        return __builtin_bit_cast(T, a) + __builtin_bit_cast(T, b);
    }
    else
    {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
        unsigned al, bl, ah, bh;
        butterfly_pair<OFF>(static_cast<unsigned>(u), al, bl);
        butterfly_pair<OFF>(static_cast<unsigned>(u >> 32), ah, bh);
        return __builtin_bit_cast(T, (static_cast<unsigned long long>(ah) << 32) | al) +
               __builtin_bit_cast(T, (static_cast<unsigned long long>(bh) << 32) | bl);
    }
}

// Sum over the wavefront in every lane, offsets 32, 16, ... 1 in turn.
template <typename T>
__device__ __forceinline__ T wave_sum(T v)
{
    v = butterfly_add<32>(v);
    v = butterfly_add<16>(v);
    v = butterfly_add<8>(v);
    v = butterfly_add<4>(v);
    v = butterfly_add<2>(v);
    v = butterfly_add<1>(v);
    return v;
}

// wave_sum of four values at once: every lane of 16-lane row q ends with the sum
// of v[q], added in wave_sum's order.  The half and row swaps merge two values
// into one register on the way, so four sums take the instructions of little
// more than one (21 instead of 112 in FP64).
template <int OFF, typename T>
__device__ __forceinline__ T butterfly_merge(T a, T b)
{
    static_assert((OFF == 32 || OFF == 16) && (sizeof(T) == 4 || sizeof(T) == 8), "lane swap");
    auto swap = [](unsigned x, unsigned y) {
        if constexpr (OFF == 32) return __builtin_amdgcn_permlane32_swap(x, y, false, false);
        else return __builtin_amdgcn_permlane16_swap(x, y, false, false);
    };
    if constexpr (sizeof(T) == 4)
    {
        const auto both = swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b));
        return __builtin_bit_cast(T, static_cast<unsigned>(both[0])) + __builtin_bit_cast(T, static_cast<unsigned>(both[1]));
    }
    else
    {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, a);
        const unsigned long long w = __builtin_bit_cast(unsigned long long, b);
        const auto lo = swap(static_cast<unsigned>(u), static_cast<unsigned>(w));
        const auto hi = swap(static_cast<unsigned>(u >> 32), static_cast<unsigned>(w >> 32));
        return __builtin_bit_cast(T, (static_cast<unsigned long long>(hi[0]) << 32) | lo[0]) +
               __builtin_bit_cast(T, (static_cast<unsigned long long>(hi[1]) << 32) | lo[1]);
    }
}

template <typename T>
__device__ __forceinline__ T wave_sum4(T v0, T v1, T v2, T v3)
{
    T v = butterfly_merge<16>(butterfly_merge<32>(v0, v2), butterfly_merge<32>(v1, v3));
    v = butterfly_add<8>(v);
    v = butterfly_add<4>(v);
    v = butterfly_add<2>(v);
    v = butterfly_add<1>(v);
    return v;
}

// Sum within aligned groups of L lanes (L a power of two <= 64); every lane of
// the group ends with the group sum.  Fixed butterfly order.
template <int L, typename T>
__device__ __forceinline__ T group_sum(T v)
{
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, kWave);
    return v;
}

// Workgroup sum of NV doubles; result valid in thread 0.  `lds` needs
// NV * (blockDim/64) doubles.
template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* lds)
{
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int waves = blockDim.x / kWave;
    if constexpr (NV == 3 || NV == 4)
    {
        const double sum = wave_sum4(v[0], v[1], v[2], v[NV - 1]);
        if (lane % 16 == 0 && lane / 16 < NV) lds[lane / 16 * 16 + wave] = sum;
    }
    else
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
        if (lane == 0)
        {
#pragma unroll
            for (int k = 0; k < NV; ++k) lds[k * 16 + wave] = v[k];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int k = 0; k < NV; ++k)
        {
            double s = 0.0;
            for (int w = 0; w < waves; ++w) s += lds[k * 16 + w];
            v[k] = s;
        }
    }
}

// Publish this workgroup's NV partial sums; the last workgroup to arrive sums
// all partials in index order (so the result does not depend on arrival order)
// and returns true in every one of its threads, with the totals in `total`
// (valid in all threads of that workgroup).  `counter` returns to zero.
template <int NV>
__device__ __forceinline__ bool last_block_total(double (&v)[NV], double* partials, unsigned* counter,
                                                 double (&total)[NV])
{
    __shared__ double lds[NV * 16];
    __shared__ int is_last;
    __shared__ double result[NV];
    const int nblocks = gridDim.x;
    block_sum<NV>(v, lds);
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) partials[k * kMaxPartials + blockIdx.x] = v[k];
        __threadfence();
        const unsigned arrived = atomicAdd(counter, 1u);
        is_last = (arrived == static_cast<unsigned>(nblocks - 1));
    }
    __syncthreads();
    if (!is_last) return false;
    __threadfence();
    double acc[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k)
    {
        double s = 0.0;
        for (int b = threadIdx.x; b < nblocks; b += blockDim.x)
            s += partials[k * kMaxPartials + b];
        acc[k] = s;
    }
    __syncthreads();
    block_sum<NV>(acc, lds);
    if (threadIdx.x == 0)
    {
#pragma unroll
        for (int k = 0; k < NV; ++k) result[k] = acc[k];
        *counter = 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) total[k] = result[k];
    return true;
}

// ---- grow-only device buffer ---------------------------------------------
struct DeviceBuffer
{
    void* ptr = nullptr;
    size_t bytes = 0;
    int reserve(size_t need);
    void release();
    template <typename T>
    T* as() const
    {
        return static_cast<T*>(ptr);
    }
};

__host__ __device__ inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

} // namespace pm
