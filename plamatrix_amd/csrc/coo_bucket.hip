// COO -> CSR by row ranges (coo_bucket.hpp).
//
// The LSD sort of coo.hip moves every triplet once per 8 key bits: five passes of
// 12 bytes read twice and written once for a million-row matrix, each pass with a
// histogram and a scan of its own.  Rows are the high key bits, so one stable
// partition by row range already leaves independent pieces, and a piece of a few
// thousand triplets sorts in LDS:
//
//   pack       keys (row << cb | col), per-tile counts of the buckets
//   columns    per bucket, the counts of the tiles before each tile
//   partition  every triplet as one 64-bit word, local key above position, to its
//              bucket, input order kept
//   sort       a workgroup per bucket: stable 8-bit passes in LDS, distinct keys
//              counted
//   runs       exclusive scan of the counts, the nnz to the host
//   fold       (finish) a workgroup per bucket: values gathered, each run summed left
//              to right by the lane of its head, row offsets by searching the
//              bucket's heads in LDS
//
// Measured, both calls together, LSD sort / here: 10,903 FP32 triplets of a 2,025-row
// stencil 143 / 65 us (18 launches and two copies / 7 launches); 5.76 M FP64
// triplets of a million rows 898 / 382 us, of them fold 125, sort 93, partition 75,
// pack 32.
//
// Up to kBucketOne triplets with at most 32 key bits are one bucket: no partition.
// Equal keys keep their input order at every step, so the result is the LSD path's.
#include "coo_bucket.hpp"

#include <algorithm>
#include <cmath>

#include "pm_common.hpp"
#include "sort.hpp"

namespace pm
{
namespace
{

typedef unsigned long long u64;

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / kWave;
constexpr int kItems = kBucketCap / kThreads;  // triplets per lane, at most

struct Tables
{
    unsigned* totals;    // [buckets]
    unsigned* base;      // [buckets + 1] first triplet of a bucket
    unsigned* heads;     // [buckets] distinct keys
    unsigned* run_base;  // [buckets + 1] first run of a bucket
    unsigned* invalid;   // [tiles][2] lowest offending positions
    unsigned* hist;      // [tiles][buckets]
};

__host__ __device__ inline size_t table_words(const CooPlan& p)
{
    return 4 * (static_cast<size_t>(p.buckets) + 64) + 2 * static_cast<size_t>(p.tiles) + 64 +
           static_cast<size_t>(p.tiles) * p.buckets;
}

Tables tables(const CooBuckets& b)
{
    Tables t{};
    const size_t step = static_cast<size_t>(b.plan.buckets) + 64;
    t.totals = reinterpret_cast<unsigned*>(b.tables);
    t.base = t.totals + step;
    t.heads = t.base + step;
    t.run_base = t.heads + step;
    t.invalid = t.run_base + step;
    t.hist = t.invalid + 2 * b.plan.tiles + 64;
    return t;
}

// Exclusive scan over the workgroup; `lds` holds kWaves + 1 words.
__device__ __forceinline__ unsigned scan_threads(unsigned v, unsigned* lds, unsigned& total)
{
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    unsigned x = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1)
    {
        const unsigned y = __shfl_up(x, off, kWave);
        if (lane >= off) x += y;
    }
    if (lane == kWave - 1) lds[wave] = x;
    __syncthreads();
    if (wave == 0)
    {
        const unsigned w = lane < kWaves ? lds[lane] : 0u;
        unsigned s = w;
#pragma unroll
        for (int off = 1; off < kWaves; off <<= 1)
        {
            const unsigned y = __shfl_up(s, off, kWave);
            if (lane >= off) s += y;
        }
        if (lane < kWaves) lds[lane] = s - w;
        if (lane == kWaves - 1) lds[kWaves] = s;
    }
    __syncthreads();
    const unsigned out = lds[wave] + x - v;
    total = lds[kWaves];
    __syncthreads();
    return out;
}

template <typename S>
__device__ __forceinline__ u64 pack_one(int64_t i, int64_t rows, int64_t cols, int cb, const int64_t* r,
                                        const int64_t* c, const S* v, int check_finite, unsigned* invalid)
{
    const int64_t row = r[i], col = c[i];
    if (check_finite && !isfinite(static_cast<double>(v[i]))) atomicMin(&invalid[1], static_cast<unsigned>(i));
    if (row >= 0 && row < rows && col >= 0 && col < cols) return (static_cast<u64>(row) << cb) | static_cast<u64>(col);
    atomicMin(&invalid[0], static_cast<unsigned>(i));
    return ~0ull;
}

__device__ __forceinline__ u64 position_or_none(unsigned p) { return p == ~0u ? ~0ull : static_cast<u64>(p); }

// Bound by reading the triplets: 24 bytes each (FP64) and 8 written.
template <typename S>
__global__ __launch_bounds__(kThreads) void k_bucket_pack(CooBuckets b, Tables t, const int64_t* __restrict__ r,
                                                          const int64_t* __restrict__ c, const S* __restrict__ v,
                                                          int check_finite)
{
    extern __shared__ unsigned hist[];
    __shared__ unsigned invalid[2];
    const int tid = threadIdx.x, nb = b.plan.buckets;
    for (int d = tid; d < nb; d += kThreads) hist[d] = 0;
    if (tid < 2) invalid[tid] = ~0u;
    __syncthreads();
    const int64_t base = static_cast<int64_t>(blockIdx.x) * b.plan.rounds * kThreads;
#pragma unroll 4
    for (int k = 0; k < b.plan.rounds; ++k)
    {
        const int64_t i = base + k * kThreads + tid;
        if (i >= b.count) continue;
        const u64 key = pack_one(i, b.rows, b.cols, b.plan.cb, r, c, v, check_finite, invalid);
        b.keys[i] = key;
        if (key != ~0ull) atomicAdd(&hist[key >> (b.plan.cb + b.plan.shift)], 1u);
    }
    __syncthreads();
    for (int d = tid; d < nb; d += kThreads) t.hist[static_cast<int64_t>(blockIdx.x) * nb + d] = hist[d];
    if (tid < 2) t.invalid[2 * blockIdx.x + tid] = invalid[tid];
}

// Per bucket the counts of the tiles before each tile, in place: a workgroup for
// 64 buckets, a wavefront for a sixteenth of the tiles.
__global__ __launch_bounds__(kThreads) void k_bucket_columns(CooBuckets b, Tables t)
{
    __shared__ unsigned part[kWaves][kWave];
    __shared__ unsigned low[2];
    const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, nb = b.plan.buckets;
    const int d = blockIdx.x * kWave + lane;
    const int64_t per = (b.plan.tiles + kWaves - 1) / kWaves;
    const int64_t from = wave * per, to = min(from + per, b.plan.tiles);
    unsigned sum = 0;
    if (d < nb)
#pragma unroll 8
        for (int64_t i = from; i < to; ++i) sum += t.hist[i * nb + d];
    part[wave][lane] = sum;
    if (threadIdx.x < 2) low[threadIdx.x] = ~0u;
    __syncthreads();
    unsigned run = 0, total = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
    {
        const unsigned s = part[w][lane];
        run += w < wave ? s : 0u;
        total += s;
    }
    if (d < nb)
    {
        if (wave == 0) t.totals[d] = total;
#pragma unroll 8
        for (int64_t i = from; i < to; ++i)
        {
            const unsigned s = t.hist[i * nb + d];
            t.hist[i * nb + d] = run;
            run += s;
        }
    }
    if (blockIdx.x != 0) return;
    unsigned a = ~0u, f = ~0u;
    for (int64_t i = threadIdx.x; i < b.plan.tiles; i += kThreads)
    {
        a = min(a, t.invalid[2 * i]);
        f = min(f, t.invalid[2 * i + 1]);
    }
    if (a != ~0u) atomicMin(&low[0], a);
    if (f != ~0u) atomicMin(&low[1], f);
    __syncthreads();
    if (threadIdx.x != 0) return;
    b.status->invalid_source = position_or_none(low[0]);
    b.status->invalid_value = position_or_none(low[1]);
    b.status->expected_nnz = -1;
    b.status->nnz = 0;
    b.status->unsorted = 0;
    b.status->most = 0;
}

// One 64-bit word per triplet, written in the order of the input within a bucket.
// A tile of 8 x 1,024 triplets puts four neighbouring words into a bucket of the
// largest conversions, half a cache line.
__global__ __launch_bounds__(kThreads) void k_bucket_partition(CooBuckets b, Tables t, int bits)
{
    extern __shared__ unsigned lds[];
    __shared__ unsigned scan[kWaves + 1];
    __shared__ int over;
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, nb = b.plan.buckets;
    const int64_t base = static_cast<int64_t>(blockIdx.x) * b.plan.rounds * kThreads;
    unsigned* start = lds;
    unsigned short* count = reinterpret_cast<unsigned short*>(lds + nb);  // [kWaves][nb]
    if (tid == 0) over = b.status->invalid_source != ~0ull;
    for (int l = tid; l < nb * kWaves / 2; l += kThreads) lds[nb + l] = 0;
    __syncthreads();
    constexpr int per = kBucketsMost / kThreads;
    unsigned mine[per], sum = 0, total;
#pragma unroll
    for (int j = 0; j < per; ++j)
    {
        mine[j] = tid * per + j < nb ? t.totals[tid * per + j] : 0u;
        sum += mine[j];
        if (mine[j] > kBucketCap) over = 1;
    }
    unsigned run = scan_threads(sum, scan, total);
#pragma unroll
    for (int j = 0; j < per; ++j)
    {
        const int d = tid * per + j;
        if (d < nb)
        {
            start[d] = run + t.hist[static_cast<int64_t>(blockIdx.x) * nb + d];
            if (blockIdx.x == 0) t.base[d] = run;
        }
        run += mine[j];
    }
    if (blockIdx.x == 0 && tid == 0) t.base[nb] = total;
    if (over)
    {
        if (blockIdx.x == 0 && tid == 0) b.status->unsorted = 1;
        return;
    }
    u64 key[kItems];
    unsigned rank[kItems];
    const int first = wave * kWave * b.plan.rounds + lane;
    const int64_t left = b.count - base;
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        key[k] = k < b.plan.rounds && first + k * kWave < left ? b.keys[base + first + k * kWave] : ~0ull;
    const int down = b.plan.cb + b.plan.shift;
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (k < b.plan.rounds)
            rank[k] = wave_rank(key[k] != ~0ull, static_cast<unsigned>(key[k] >> down) & ((1u << bits) - 1u), bits,
                                count + wave * nb);
    __syncthreads();
    for (int d = tid; d < nb; d += kThreads)
    {
        unsigned before = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w)
        {
            const unsigned n = count[w * nb + d];
            count[w * nb + d] = static_cast<unsigned short>(before);
            before += n;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if (k < b.plan.rounds && key[k] != ~0ull)
        {
            const unsigned d = static_cast<unsigned>(key[k] >> down);
            const u64 local = key[k] & ((1ull << down) - 1ull);
            b.words[start[d] + count[wave * nb + d] + rank[k]] =
                (local << 32) | static_cast<unsigned>(base + first + k * kWave);
        }
}

struct SortLds
{
    u64 words[kBucketCap];
    unsigned short count[kWaves][256];
    unsigned start[256];
    unsigned scan[kWaves + 1];
    unsigned invalid[2];
    int heads;
};

// The workgroup's n words of `in` by their local keys, to `out`; sh.heads receives
// the number of distinct keys.  R: rounds, at most.
template <int R, typename Load>
__device__ __forceinline__ void sort_bucket(SortLds& sh, int n, int key_bits, Load load, u64* __restrict__ out)
{
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int rounds = (n + kThreads - 1) / kThreads;
    int first = wave * kWave * rounds + lane;
    u64 word[R];
    unsigned rank[R];
#pragma unroll
    for (int k = 0; k < R; ++k) word[k] = k < rounds && first + k * kWave < n ? load(first + k * kWave) : 0;
    for (int shift = 0; shift < key_bits; shift += 8)
    {
        asm volatile("" : "+v"(first));  // the rounds' masks are not kept over the passes
        for (int l = tid; l < kWaves * 256 / 2; l += kThreads) reinterpret_cast<unsigned*>(sh.count)[l] = 0;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k < rounds)
                rank[k] = wave_rank(first + k * kWave < n, static_cast<unsigned>(word[k] >> (32 + shift)) & 0xffu, 8,
                                    sh.count[wave]);
        __syncthreads();
        unsigned before = 0;
        if (tid < 256)
        {
#pragma unroll
            for (int w = 0; w < kWaves; ++w)
            {
                const unsigned m = sh.count[w][tid];
                sh.count[w][tid] = static_cast<unsigned short>(before);
                before += m;
            }
        }
        unsigned total;
        const unsigned at = scan_threads(before, sh.scan, total);
        if (tid < 256) sh.start[tid] = at;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k < rounds && first + k * kWave < n)
            {
                const unsigned d = static_cast<unsigned>(word[k] >> (32 + shift)) & 0xffu;
                sh.words[sh.start[d] + sh.count[wave][d] + rank[k]] = word[k];
            }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k < rounds && first + k * kWave < n) word[k] = sh.words[first + k * kWave];
    }
    if (key_bits == 0)
    {
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (k < rounds && first + k * kWave < n) sh.words[first + k * kWave] = word[k];
        __syncthreads();
    }
    int mine = 0;
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int i = first + k * kWave;
        const bool in = k < rounds && i < n;
        const bool head = in && (i == 0 || static_cast<unsigned>(sh.words[i - 1] >> 32) != static_cast<unsigned>(word[k] >> 32));
        mine += __popcll(__ballot(head));
        if (in) out[i] = word[k];
    }
    if (lane == 0 && mine != 0) atomicAdd(&sh.heads, mine);
    __syncthreads();
}

// A bucket per workgroup.  Bound by the serial passes, five barriers each: two
// workgroups share a CU, and buckets of the usual size take the body of four
// rounds, whose words and ranks fit the registers of that.
__global__ __launch_bounds__(kThreads, 8) void k_bucket_sort(CooBuckets b, Tables t)
{
    extern __shared__ char raw[];
    SortLds& sh = *reinterpret_cast<SortLds*>(raw);
    if (b.status->unsorted) return;
    const int64_t base = t.base[blockIdx.x];
    const int n = static_cast<int>(t.base[blockIdx.x + 1] - t.base[blockIdx.x]);
    if (threadIdx.x == 0) sh.heads = 0;
    const u64* in = b.words + base;
    auto load = [&](int i) { return in[i]; };
    if (n <= 4 * kThreads) sort_bucket<4>(sh, n, b.plan.cb + b.plan.shift, load, b.keys + base);
    else sort_bucket<kItems>(sh, n, b.plan.cb + b.plan.shift, load, b.keys + base);
    if (threadIdx.x == 0) t.heads[blockIdx.x] = static_cast<unsigned>(sh.heads);
}

// A conversion of one bucket, from the triplets to the status record, in one
// workgroup.
template <typename S>
__global__ __launch_bounds__(kThreads) void k_bucket_one(CooBuckets b, Tables t, const int64_t* __restrict__ r,
                                                         const int64_t* __restrict__ c, const S* __restrict__ v,
                                                         int check_finite, CooStatus* host, u64 ticket)
{
    extern __shared__ char raw[];
    SortLds& sh = *reinterpret_cast<SortLds*>(raw);
    const int tid = threadIdx.x, n = static_cast<int>(b.count);
    if (tid < 2) sh.invalid[tid] = ~0u;
    if (tid == 0) sh.heads = 0;
    __syncthreads();
    for (int i = tid; i < n; i += kThreads)
    {
        const u64 key = pack_one(static_cast<int64_t>(i), b.rows, b.cols, b.plan.cb, r, c, v, check_finite, sh.invalid);
        b.keys[i] = key;
        sh.words[i] = (key << 32) | static_cast<unsigned>(i);
    }
    __syncthreads();
    const bool valid = sh.invalid[0] == ~0u;
    auto load = [&](int i) { return sh.words[i]; };
    if (valid) sort_bucket<kItems>(sh, n, b.plan.cb + b.plan.shift, load, b.words);
    if (tid != 0) return;
    CooStatus s{};
    s.invalid_source = position_or_none(sh.invalid[0]);
    s.invalid_value = position_or_none(sh.invalid[1]);
    s.expected_nnz = -1;
    s.nnz = sh.heads;
    s.unsorted = valid ? 0 : 1;
    s.most = static_cast<u64>(n);
    *b.status = s;
    t.base[0] = 0;
    t.base[1] = static_cast<unsigned>(n);
    t.run_base[0] = 0;
    t.run_base[1] = static_cast<unsigned>(sh.heads);
    *host = s;
    __hip_atomic_store(&host->ticket, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

__global__ __launch_bounds__(kThreads) void k_bucket_runs(CooBuckets b, Tables t, CooStatus* host, u64 ticket)
{
    __shared__ unsigned scan[kWaves + 1];
    constexpr int per = kBucketsMost / kThreads;
    const int tid = threadIdx.x, nb = b.plan.buckets;
    CooStatus s = *b.status;
    s.ticket = 0;
    __shared__ unsigned most;
    if (tid == 0) most = 0;
    __syncthreads();
    if (!s.unsorted)
    {
        unsigned mine[per], sum = 0, top = 0, total;
#pragma unroll
        for (int j = 0; j < per; ++j)
        {
            mine[j] = tid * per + j < nb ? t.heads[tid * per + j] : 0u;
            sum += mine[j];
            if (tid * per + j < nb) top = max(top, t.totals[tid * per + j]);
        }
#pragma unroll
        for (int off = kWave / 2; off > 0; off /= 2) top = max(top, static_cast<unsigned>(__shfl_xor(top, off, kWave)));
        if (tid % kWave == 0) atomicMax(&most, top);
        unsigned run = scan_threads(sum, scan, total);
#pragma unroll
        for (int j = 0; j < per; ++j)
        {
            if (tid * per + j < nb) t.run_base[tid * per + j] = run;
            run += mine[j];
        }
        s.nnz = total;
        s.most = most;
        if (tid == 0)
        {
            t.run_base[nb] = total;
            b.status->nnz = s.nnz;
        }
    }
    if (tid != 0) return;
    *host = s;
    __hip_atomic_store(&host->ticket, ticket, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Bound by the gather of the values (a cache line for each, from the
// memory-side cache) and the 16 bytes written per run.
template <typename S>
__global__ __launch_bounds__(kThreads) void k_bucket_fold(CooBuckets b, Tables t, const u64* __restrict__ words,
                                                          const S* __restrict__ v, int check_finite, int64_t capacity,
                                                          int64_t* __restrict__ row_offsets, int64_t* __restrict__ cols,
                                                          S* __restrict__ vals, int most)
{
    extern __shared__ char raw[];
    struct
    {
        S* values;
        unsigned* keys;  // then the rows of the heads
    } sh;
    sh.values = reinterpret_cast<S*>(raw);
    sh.keys = reinterpret_cast<unsigned*>(sh.values + most);
    __shared__ unsigned part[kWaves];
    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int64_t base = t.base[blockIdx.x], run_base = t.run_base[blockIdx.x];
    const int n = static_cast<int>(t.base[blockIdx.x + 1] - t.base[blockIdx.x]);
    const int heads = static_cast<int>(t.run_base[blockIdx.x + 1] - t.run_base[blockIdx.x]);
    const int rounds = (n + kThreads - 1) / kThreads;
    const int first = wave * kWave * rounds + lane, cb = b.plan.cb;
    u64 word[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k)
    {
        const int i = first + k * kWave;
        word[k] = k < rounds && i < n ? words[base + i] : 0;
    }
#pragma unroll
    for (int k = 0; k < kItems; ++k)
    {
        const int i = first + k * kWave;
        if (k >= rounds || i >= n) continue;
        sh.values[i] = v[static_cast<unsigned>(word[k])];
        sh.keys[i] = static_cast<unsigned>(word[k] >> 32);
    }
    __syncthreads();
    u64 head[kItems];
    unsigned mine = 0;
#pragma unroll
    for (int k = 0; k < kItems; ++k)
    {
        const int i = first + k * kWave;
        const bool in = k < rounds && i < n;
        head[k] = __ballot(in && (i == 0 || sh.keys[i - 1] != static_cast<unsigned>(word[k] >> 32)));
        mine += static_cast<unsigned>(__popcll(head[k]));
    }
    if (lane == 0) part[wave] = mine;
    __syncthreads();
    unsigned run = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) run += w < wave ? part[w] : 0u;
    unsigned at[kItems];
#pragma unroll
    for (int k = 0; k < kItems; ++k)
    {
        at[k] = run + static_cast<unsigned>(__popcll(head[k] & ((1ull << lane) - 1ull)));
        run += static_cast<unsigned>(__popcll(head[k]));
        if (!((head[k] >> lane) & 1ull)) continue;
        const int i = first + k * kWave;
        const unsigned key = static_cast<unsigned>(word[k] >> 32);
        S sum = sh.values[i];
        if (check_finite && !isfinite(static_cast<double>(sum)))
            atomicMin(&b.status->invalid_value, static_cast<u64>(static_cast<unsigned>(word[k])));
        for (int j = i + 1; j < n && sh.keys[j] == key; ++j)
        {
            sum += sh.values[j];
            if (check_finite && !isfinite(static_cast<double>(sum)))
                atomicMin(&b.status->invalid_value, static_cast<u64>(static_cast<unsigned>(words[base + j])));
        }
        const int64_t to = run_base + at[k];
        if (to < capacity)
        {
            cols[to] = static_cast<int64_t>(static_cast<u64>(key) & ((1ull << cb) - 1ull));
            vals[to] = sum;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kItems; ++k)
        if ((head[k] >> lane) & 1ull) sh.keys[at[k]] = static_cast<unsigned>((word[k] >> 32) >> cb);
    __syncthreads();
    // row offsets of the bucket's rows: heads of smaller rows, by binary search
    const int64_t row0 = static_cast<int64_t>(blockIdx.x) << b.plan.shift;
    const int64_t row1 = min(row0 + (static_cast<int64_t>(1) << b.plan.shift), b.rows);
    for (int64_t row = row0 + tid; row < row1; row += kThreads)
    {
        int lo = 0, hi = heads;
        while (lo < hi)
        {
            const int mid = (lo + hi) / 2;
            if (sh.keys[mid] < static_cast<unsigned>(row - row0)) lo = mid + 1;
            else hi = mid;
        }
        row_offsets[row] = min(run_base + lo, capacity);
    }
    if (tid != 0) return;
    if (blockIdx.x == gridDim.x - 1) row_offsets[b.rows] = min(run_base + heads, capacity);
    if (blockIdx.x == 0) b.status->expected_nnz = capacity;
}

__global__ __launch_bounds__(kThreads) void k_bucket_unpack(CooBuckets b, Tables t, unsigned* __restrict__ positions)
{
    if (b.plan.tiles == 0 || b.status->unsorted)
    {
        for (int64_t i = static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x; i < b.count;
             i += static_cast<int64_t>(gridDim.x) * kThreads)
            positions[i] = static_cast<unsigned>(i);
        return;
    }
    for (int d = blockIdx.x; d < b.plan.buckets; d += gridDim.x)
    {
        const u64 high = static_cast<u64>(d) << (b.plan.cb + b.plan.shift);
        for (int64_t i = t.base[d] + threadIdx.x; i < t.base[d + 1]; i += kThreads)
        {
            const u64 word = b.keys[i];
            b.keys[i] = high | (word >> 32);
            positions[i] = static_cast<unsigned>(word);
        }
    }
}

// `bytes`: the most that any conversion asks of the kernel (the limit belongs to the
// process, and another thread's conversion may need more than this one).
template <typename K>
int allow_lds(K kernel, size_t bytes)
{
    PM_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               static_cast<int>(bytes)));
    return PM_OK;
}

} // namespace

// Buckets of 2^shift rows, the most that keep the mean at kBucketMean and a local
// key in 32 bits (and kBucketRowBits): uneven rows may then be 2.7 times the mean
// before a bucket outgrows its workgroup (the conversion then pays the partition's
// counts and goes on in the LSD sort: 100,000 triplets 184 us against 154 by the sort
// alone, 5.76 M 752 against 700).  Longer rows, wider keys and more than kBucketsMost
// buckets stay on the LSD sort.
//
// Smaller conversions are cut finer, towards a bucket per CU but not below
// kBucketMeanLeast: the passes of a bucket are serial (10,939 triplets as 22 buckets
// 65 us, as 4 70; 89,549 68 against 74; no difference from 400,000 on).  One bucket
// without a partition is level with several at 4,200 to 5,000 triplets (4,189: 61.5
// against 62.4 us; 5,491: 65.1 against 63.0).
CooPlan coo_plan(int64_t rows, int64_t cols, int64_t count)
{
    CooPlan p{};
    const int rb = bits_for(rows), cb = bits_for(cols);
    if (count <= 0 || rows <= 0 || cols <= 0 || cb > 32 || rows >= (int64_t(1) << 40)) return p;
    p.cb = cb;
    if (count <= kBucketOne && rb <= kBucketRowBits && rb + cb <= 32)
    {
        p.buckets = 1;
        p.shift = rb;
        return p;
    }
    int shift = std::min({rb, 32 - cb, kBucketRowBits});
    const double mean = static_cast<double>(
        std::min<int64_t>(kBucketMean, std::max<int64_t>(kBucketMeanLeast, count / kBucketsWanted)));
    while (shift > 0 && static_cast<double>(count) * static_cast<double>(int64_t(1) << shift) >
                            mean * static_cast<double>(rows))
        --shift;
    if (static_cast<double>(count) * static_cast<double>(int64_t(1) << shift) >
        static_cast<double>(kBucketMean) * static_cast<double>(rows))
        return p;
    const int64_t buckets = ((rows - 1) >> shift) + 1;
    if (buckets > kBucketsMost) return p;
    p.buckets = static_cast<int>(buckets);
    p.shift = shift;
    // a tile per CU until a tile is eight rounds
    p.rounds = static_cast<int>(std::min<int64_t>(kItems, std::max<int64_t>(1, count / (256 * kThreads))));
    p.tiles = ceil_div(count, static_cast<int64_t>(p.rounds) * kThreads);
    return p;
}

size_t coo_bucket_bytes(const CooPlan& plan) { return plan.buckets > 0 ? sizeof(unsigned) * table_words(plan) : 0; }

template <typename S>
int coo_bucket_prepare(const CooBuckets& b, const int64_t* r, const int64_t* c, const S* v, int check_finite,
                       CooStatus* host, unsigned long long ticket, hipStream_t stream)
{
    const Tables t = tables(b);
    const CooPlan& p = b.plan;
    if (p.tiles == 0)
    {
        auto* one = k_bucket_one<S>;
        PM_TRY(allow_lds(one, sizeof(SortLds)));
        hipLaunchKernelGGL(one, dim3(1), dim3(kThreads), sizeof(SortLds), stream, b, t, r, c, v, check_finite, host, ticket);
        PM_HIP(hipGetLastError());
        return PM_OK;
    }
    hipLaunchKernelGGL(k_bucket_pack<S>, dim3(p.tiles), dim3(kThreads), sizeof(unsigned) * p.buckets, stream, b, t, r, c,
                       v, check_finite);
    PM_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_bucket_columns, dim3(ceil_div(p.buckets, kWave)), dim3(kThreads), 0, stream, b, t);
    PM_HIP(hipGetLastError());
    constexpr size_t per_bucket = sizeof(unsigned) + sizeof(unsigned short) * kWaves;
    const size_t lds = per_bucket * p.buckets;
    PM_TRY(allow_lds(k_bucket_partition, per_bucket * kBucketsMost));
    hipLaunchKernelGGL(k_bucket_partition, dim3(p.tiles), dim3(kThreads), lds, stream, b, t, bits_for(p.buckets));
    PM_HIP(hipGetLastError());
    PM_TRY(allow_lds(k_bucket_sort, sizeof(SortLds)));
    hipLaunchKernelGGL(k_bucket_sort, dim3(p.buckets), dim3(kThreads), sizeof(SortLds), stream, b, t);
    PM_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_bucket_runs, dim3(1), dim3(kThreads), 0, stream, b, t, host, ticket);
    PM_HIP(hipGetLastError());
    return PM_OK;
}

template <typename S>
int coo_bucket_finish(const CooBuckets& b, const S* v, int check_finite, int64_t capacity, int64_t* row_offsets,
                      int64_t* cols, S* vals, int64_t most, hipStream_t stream)
{
    auto* fold = k_bucket_fold<S>;
    const int room = static_cast<int>((most + 255) / 256 * 256);
    const size_t lds = (sizeof(S) + sizeof(unsigned)) * room;
    PM_TRY(allow_lds(fold, (sizeof(S) + sizeof(unsigned)) * kBucketCap));
    hipLaunchKernelGGL(fold, dim3(b.plan.buckets), dim3(kThreads), lds, stream, b, tables(b),
                       b.plan.tiles == 0 ? b.words : b.keys, v, check_finite, capacity, row_offsets, cols, vals, room);
    PM_HIP(hipGetLastError());
    return PM_OK;
}

int coo_bucket_unpack(const CooBuckets& b, unsigned* positions, hipStream_t stream)
{
    const int64_t grid = std::max<int64_t>(b.plan.buckets, std::min<int64_t>(ceil_div(b.count, kThreads), 2048));
    hipLaunchKernelGGL(k_bucket_unpack, dim3(static_cast<unsigned>(grid)), dim3(kThreads), 0, stream, b, tables(b), positions);
    PM_HIP(hipGetLastError());
    return PM_OK;
}

template int coo_bucket_prepare<float>(const CooBuckets&, const int64_t*, const int64_t*, const float*, int, CooStatus*,
                                       unsigned long long, hipStream_t);
template int coo_bucket_prepare<double>(const CooBuckets&, const int64_t*, const int64_t*, const double*, int, CooStatus*,
                                        unsigned long long, hipStream_t);
template int coo_bucket_finish<float>(const CooBuckets&, const float*, int, int64_t, int64_t*, int64_t*, float*, int64_t,
                                       hipStream_t);
template int coo_bucket_finish<double>(const CooBuckets&, const double*, int, int64_t, int64_t*, int64_t*, double*, int64_t,
                                        hipStream_t);

} // namespace pm
