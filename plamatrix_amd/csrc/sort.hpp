// Device scan and stable radix sort shared by COO -> CSR and the Schur
// pattern / normal-equation topology builders.
#pragma once

#include "pm_common.hpp"

namespace pm
{

// Exclusive scan of n u32 values (in may equal out); `grand_total` (device,
// may be null) receives the sum.  `scratch` holds scan_scratch_words(n) words.
int64_t scan_scratch_words(int64_t n);
int scan_u32(const unsigned* in, unsigned* out, int64_t n, unsigned* scratch, unsigned* grand_total,
             hipStream_t stream);

// Stable LSD radix sort of (key, value) pairs on the low key_bits bits, 8 bits
// per pass.  The input is in keys_a / vals_a; the sorted result ends in the
// b buffers when *in_b is set, else in the a buffers.  `hist` holds
// radix_hist_words(count) words and `scratch` scan_scratch_words of that.
int radix_sort_pairs(unsigned long long* keys_a, unsigned* vals_a, unsigned long long* keys_b, unsigned* vals_b,
                     int64_t count, int key_bits, unsigned* hist, unsigned* scratch, hipStream_t stream, bool* in_b);
int64_t radix_hist_words(int64_t count);

// Smallest b with 2^b >= n.
int bits_for(int64_t n);

// Rank of an active lane among the wavefront's earlier occurrences of its digit,
// by ballots; `count`: the wavefront's running count per digit.  Lanes of a
// wavefront run in step, so every lane reads the count before the first lane of
// its digit raises it.
__device__ __forceinline__ unsigned wave_rank(bool active, unsigned digit, int bits, unsigned short* count)
{
    unsigned long long peers = __ballot(active);
    for (int bit = 0; bit < bits; ++bit)
    {
        const unsigned long long ones = __ballot((digit >> bit) & 1u);
        peers &= ((digit >> bit) & 1u) ? ones : ~ones;
    }
    const unsigned below = static_cast<unsigned>(__popcll(peers & ((1ull << (threadIdx.x % kWave)) - 1ull)));
    const unsigned before =
        active ? __hip_atomic_load(count + digit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT) : 0u;
    __builtin_amdgcn_wave_barrier();
    if (active && below == 0)
        __hip_atomic_store(count + digit, static_cast<unsigned short>(before + __popcll(peers)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_WAVEFRONT);
    __builtin_amdgcn_sched_barrier(0);  // one round's ballots at a time
    return before + below;
}

} // namespace pm
