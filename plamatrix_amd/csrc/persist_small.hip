// A whole single-reduction CG / Jacobi-PCG solve of a small CSR matrix in one
// workgroup.
//
// Below a few thousand rows an iteration of two kernels is nothing but kernel
// boundaries (1,665 rows: 13.8 us per iteration, 8 us of it inside the kernels).
// Here one workgroup of 1,024 threads runs the solve: p, s, x, r, w and the
// first entries of every row in registers, u in LDS, and two workgroup barriers
// per phase instead of launches; rows longer than the register entries read the
// rest from the caches.
//
// The dot products are summed in the order of the per-kernel iteration (the
// rows of each of its workgroups by wavefront, the workgroups by slot) and rows
// are walked left to right as its SpMV walks them, so a solve is bitwise the
// per-kernel solve.  That SpMV switches to several lanes per row in a 64-row
// chunk of more than kMaxWindows * kStreamCap entries; a matrix with such a
// chunk is left to it.
#include "persist.hpp"

#include "persist_launch.hpp"
#include "spmv_kernels.hpp"
#include "tuning.hpp"

namespace pm
{
namespace
{

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
constexpr int kSmallGroups = kSmallThreads / kBlock;  // per-kernel workgroups handled at a time
constexpr int64_t kSmallRows = 4096;                  // four rows per lane
// entries beyond the registers come from the L2 at about 64 bytes per clock of
// the one CU: 32,768 entries of 16 bytes take as long as the two kernels
constexpr int64_t kSmallEntries = 32768;
// FP64 with four rows per lane spills (108 to 137 registers of a lane): 3 entries a row
// on average 12.6 us per iteration in the two kernels against 10.4 here (4,000 rows,
// scattered columns), 5 entries 13.3 against 14.0, 7 entries 13.7 against 16.9.  A
// 5-point stencil (7.9 here at 2,116 rows, 8.0 at 4,096) takes 5.8 with a row per lane
// (persist_csr.hip).
constexpr int64_t kSmallSpillRows = 2048;
constexpr int64_t kSmallSpillEntries = 4;  // a row
constexpr int64_t kSmallSegment = 65536;              // iterations per launch
constexpr unsigned kSmallDone = 1, kSmallUnsupported = 2;

template <typename S, typename I>
struct SmallArgs
{
    int rows;
    const I* ro;
    const I* ci;
    const S* values;
    S *x, *p, *r, *s, *w, *u;
    const S* inv;
    const S* rhs;
    SolverState* st;
    double* region;
    int count, per, refresh, t0, t_end, chunk, grow;
};

template <typename S, typename I, int R, bool JACOBI>
__global__ __launch_bounds__(kSmallThreads) void k_cg_small(SmallArgs<S, I> a)
{
    constexpr int E = sizeof(S) == 8 ? 5 : 8;  // row entries in registers
    constexpr int NV = JACOBI ? 4 : 3;
    constexpr int kSlots = R * kSmallGroups;   // per-kernel workgroups at most
    __shared__ S us[R * kSmallThreads];
    __shared__ double lds_p[kCgValues][R][kSmallWaves];
    __shared__ S sh_alpha, sh_beta;
    __shared__ int sh_code, sh_long;
    __shared__ PersistHistory hs;

    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int grp = tid / kBlock, gwave = wave % kWavesPerBlock;
    const int rows = a.rows;
    if (tid == 0) sh_long = 0;
    __syncthreads();
    // 64-row chunks that the per-kernel SpMV would not walk lane by lane
    for (int c = tid; c * kChunkRows < rows; c += kSmallThreads)
    {
        const int last = (c + 1) * kChunkRows < rows ? (c + 1) * kChunkRows : rows;
        if (static_cast<int64_t>(a.ro[last]) - static_cast<int64_t>(a.ro[c * kChunkRows]) > kMaxWindows * kStreamCap)
            sh_long = 1;
    }
    __syncthreads();
    if (sh_long != 0)
    {
        if (tid == 0) a.st->counters[kCounterOutcome] = kSmallUnsupported;
        return;
    }

    // rows of the lane: slot k is row `gwave`, `lane` of logical workgroup
    // grp + k * kSmallGroups
    S p[R], s[R], x[R], r[R], w[R], inv[R], val[R][E];
    int first[R], rest[R], end[R];  // row, entries beyond the registers
    unsigned short col[R][E];
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int i = ((grp + k * kSmallGroups) * a.per + gwave) * kChunkRows + lane;
        const bool ok = gwave < a.per && grp + k * kSmallGroups < a.count && i < rows;
        first[k] = ok ? i : -1;
        const int at = ok ? i : 0;
        p[k] = ok ? a.p[at] : S(0);
        s[k] = ok ? a.s[at] : S(0);
        x[k] = ok ? a.x[at] : S(0);
        r[k] = ok ? a.r[at] : S(0);
        w[k] = ok ? a.w[at] : S(0);
        inv[k] = JACOBI && ok ? a.inv[at] : S(0);
        const int64_t b = static_cast<int64_t>(a.ro[at]);
        const int n = ok ? static_cast<int>(static_cast<int64_t>(a.ro[at + 1]) - b) : 0;
#pragma unroll
        for (int e = 0; e < E; ++e)
        {
            // an absent entry is 0 times the row's own u, which keeps the bits
            // of a finite sum
            val[k][e] = e < n ? a.values[b + e] : S(0);
            col[k][e] = static_cast<unsigned short>(e < n ? static_cast<int>(a.ci[b + e]) : at);
        }
        rest[k] = static_cast<int>(b) + (n < E ? n : E);
        end[k] = static_cast<int>(b) + n;
    }
    if (tid == 0) hs.begin(a.st, a.t_end);
    auto u_of = [&](int k) { return JACOBI ? inv[k] * r[k] : r[k]; };
    // acc[k] = row k of A v for the v in us, entries left to right
    auto product = [&](auto* acc) {
        using Acc = std::remove_reference_t<decltype(acc[0])>;
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            Acc sum = Acc(0);
#pragma unroll
            for (int e = 0; e < E; ++e)
                sum = fma_s<Acc>(static_cast<Acc>(val[k][e]), static_cast<Acc>(us[col[k][e]]), sum);
            for (int q = rest[k]; q < end[k]; ++q)
                sum = fma_s<Acc>(static_cast<Acc>(a.values[q]), static_cast<Acc>(us[a.ci[q]]), sum);
            acc[k] = sum;
        }
    };
    // sums of the partials (entry b: per-kernel workgroup b) by wavefront 0,
    // as reduce_partials_at adds them
    auto entry = [&](int v, int b) {
        const int lb = static_cast<int>(xcd_logical_block(b, a.count));
        const int q = lb % kSmallGroups, k = lb / kSmallGroups;
        double sum = 0.0;
#pragma unroll
        for (int z = 0; z < kWavesPerBlock; ++z) sum += lds_p[v][k][q * kWavesPerBlock + z];
        return sum;
    };

    int code = kRunning;
    for (int t = a.t0;; ++t)
    {
        __syncthreads();
        if (wave == 0)
        {
            // row v of the wavefront sums value v: lane j takes entry j, the
            // butterfly's first two offsets would only add the absent slots
            // from 16 on
            static_assert(kSlots <= 16, "a row of lanes reduces the partials");
            const int v = lane / 16, b = lane % 16;
            double e = 0.0;
            if (v < NV && b < a.count)
                e += t == a.t0 ? a.region[(!JACOBI && v > 0 ? v + 1 : v) * kMaxPartials + b] : entry(v, b);
            e = butterfly_add<8>(e);
            e = butterfly_add<4>(e);
            e = butterfly_add<2>(e);
            e = butterfly_add<1>(e);
            double tot[NV];
#pragma unroll
            for (int q = 0; q < NV; ++q) tot[q] = __shfl(e, q * 16, kWave);
            if (lane == 0)
                sh_code = hs.decide<S>(t, tot[0], tot[JACOBI ? 1 : 0], tot[NV - 2], tot[NV - 1], a.chunk, a.grow != 0,
                                       sh_alpha, sh_beta);
        }
        __syncthreads();
        code = sh_code;
        if (code != kRunning) break;
        const S al = sh_alpha, be = sh_beta;
        const bool refresh = a.refresh > 0 && (t + 1) % a.refresh == 0;
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            p[k] = fma_s(be, p[k], u_of(k));
            s[k] = fma_s(be, s[k], w[k]);
            x[k] = fma_s(al, p[k], x[k]);
            if (!refresh) r[k] = fma_s(-al, s[k], r[k]);
        }
        if (refresh)
        {
            // r = b - A x with FP64 accumulation
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (first[k] >= 0) us[first[k]] = x[k];
            __syncthreads();
            double ax[R];
            product(ax);
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (first[k] >= 0) r[k] = static_cast<S>(static_cast<double>(a.rhs[first[k]]) - ax[k]);
            __syncthreads();
        }
#pragma unroll
        for (int k = 0; k < R; ++k)
            if (first[k] >= 0) us[first[k]] = u_of(k);
        __syncthreads();
        product(w);
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            if (first[k] < 0) w[k] = S(0);
            const double rv = static_cast<double>(r[k]), uv = static_cast<double>(u_of(k));
            double part[kCgValues];
            part[0] = __builtin_fma(rv, rv, 0.0);
            if (JACOBI) part[1] = __builtin_fma(rv, uv, 0.0);
            part[NV - 2] = __builtin_fma(static_cast<double>(w[k]), uv, 0.0);
            part[NV - 1] = __builtin_fma(uv, static_cast<double>(s[k]), 0.0);
            const double sum = wave_sum4(part[0], part[1], part[2], part[NV - 1]);
            if (lane % 16 == 0) lds_p[lane / 16][k][wave] = sum;
        }
    }

    const bool over = code == kHandOver;
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int i = first[k];
        if (i < 0) continue;
        a.x[i] = x[k];
        if (!over) continue;
        a.p[i] = p[k];
        a.s[i] = s[k];
        a.r[i] = r[k];
        a.w[i] = w[k];
        if (JACOBI) a.u[i] = u_of(k);
    }
    if (over && tid < a.count)
    {
        // t0 and the hand-over iteration are even: the last partials are of an
        // odd iteration, region 1
        a.region[tid] = entry(0, tid);
        a.region[kMaxPartials + tid] = entry(JACOBI ? 1 : 0, tid);
        a.region[2 * kMaxPartials + tid] = entry(NV - 2, tid);
        a.region[3 * kMaxPartials + tid] = entry(NV - 1, tid);
    }
    if (tid == 0)
    {
        hs.record(a.st, code);
        a.st->counters[kCounterOutcome] = kSmallDone;
    }
}

template <typename S, typename I>
const void* small_kernel(int slots, bool jacobi)
{
    if (slots <= 1)
        return jacobi ? reinterpret_cast<const void*>(k_cg_small<S, I, 1, true>)
                      : reinterpret_cast<const void*>(k_cg_small<S, I, 1, false>);
    if (slots <= 2)
        return jacobi ? reinterpret_cast<const void*>(k_cg_small<S, I, 2, true>)
                      : reinterpret_cast<const void*>(k_cg_small<S, I, 2, false>);
    return jacobi ? reinterpret_cast<const void*>(k_cg_small<S, I, 4, true>)
                  : reinterpret_cast<const void*>(k_cg_small<S, I, 4, false>);
}

template <typename S, typename I>
int small_run(pm_workspace* ws, const PersistProblem& p, const I* ro, const I* ci, int64_t max_iterations,
              hipStream_t stream, int* outcome, int64_t* next, SolverState* state)
{
    SmallArgs<S, I> a{};
    a.rows = static_cast<int>(p.rows);
    a.ro = ro;
    a.ci = ci;
    a.values = static_cast<const S*>(p.a->values);
    a.x = static_cast<S*>(p.x);
    a.p = static_cast<S*>(p.p);
    a.r = static_cast<S*>(p.r);
    a.s = static_cast<S*>(p.s);
    a.w = static_cast<S*>(p.w);
    a.u = static_cast<S*>(p.u);
    a.inv = static_cast<const S*>(p.inv);
    a.rhs = static_cast<const S*>(p.rhs);
    a.st = p.st;
    a.region = p.region;
    a.count = p.count;
    a.per = static_cast<int>(ceil_div(chunk_count(p.rows), static_cast<int64_t>(p.count)));
    a.refresh = p.refresh;
    a.chunk = p.chunk;
    a.grow = p.grow ? 1 : 0;
    const void* kernel = small_kernel<S, I>(static_cast<int>(ceil_div(p.count, kSmallGroups)), p.jacobi);
    *outcome = kPersistAbandoned;
    const int64_t segment = persist_segment(kSmallSegment);
    for (int64_t t = 0;;)
    {
        // an even number of iterations, the last one's decision included
        const int64_t left = max_iterations + 2 - t;
        a.t0 = static_cast<int>(t);
        a.t_end = static_cast<int>(t + std::min<int64_t>(segment, left + (left & 1)));
        void* args[] = {&a};
        PM_HIP(hipLaunchKernel(kernel, dim3(1), dim3(kSmallThreads), args, 0, stream));
        PM_HIP(hipMemcpyAsync(ws->host_state, p.st, sizeof(SolverState), hipMemcpyDeviceToHost, stream));
        PM_HIP(hipStreamSynchronize(stream));
        *state = ws->host_state[0];
        if (state->counters[kCounterOutcome] != kSmallDone) return PM_OK;
        if (state->done != kRunning)
        {
            *outcome = kPersistStopped;
            return PM_OK;
        }
        t = static_cast<int64_t>(state->counters[kCounterNext]);
        if (state->counters[kCounterRestart] != 0u)
        {
            *outcome = kPersistHandOver;
            *next = t;
            return PM_OK;
        }
    }
}

} // namespace

bool persist_small_wanted(const PersistProblem& p)
{
    // one row per lane and slot: the per-kernel workgroups hold at most four
    // chunks of 64 rows
    const bool spills = p.dtype == PM_F64 && p.rows > kSmallSpillRows;
    return persist_enabled() && p.rows > 0 && p.rows <= kSmallRows && p.a->nnz <= kSmallEntries &&
           (!spills || p.a->nnz <= kSmallSpillEntries * p.rows) && p.count <= 4 * kSmallGroups && ceil_div(chunk_count(p.rows), static_cast<int64_t>(p.count)) <= kWavesPerBlock;
}

int persist_small_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                      int* outcome, int64_t* next, SolverState* state)
{
    const bool compact = use_compact(p.a);
    if (p.dtype == PM_F64)
        return compact ? small_run<double>(ws, p, p.a->row_offsets32, p.a->col_indices32, max_iterations, stream,
                                           outcome, next, state)
                       : small_run<double>(ws, p, p.a->row_offsets, p.a->col_indices, max_iterations, stream, outcome,
                                           next, state);
    return compact ? small_run<float>(ws, p, p.a->row_offsets32, p.a->col_indices32, max_iterations, stream, outcome,
                                      next, state)
                   : small_run<float>(ws, p, p.a->row_offsets, p.a->col_indices, max_iterations, stream, outcome, next,
                                      state);
}

} // namespace pm
