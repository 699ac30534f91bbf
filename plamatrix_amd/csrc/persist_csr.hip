// The persistent solve (persist.hip) for CSR matrices of short, mostly local rows:
// a row per lane, its vectors in registers and its entries in LDS.
//
// Between the sizes of one workgroup (persist_small.hip) and the diagonal layout
// an iteration of two kernels costs 11 to 14 us, nearly all of it kernel
// boundaries.  Here an entry whose column lies in the workgroup's own 1,024 rows
// reads u from LDS; any other reads the tagged word its owner published, all of
// a row's in flight at once.  Rows are walked left to right and the dot products
// summed as the per-kernel iteration does, so a solve is bitwise the same.
//
// Words of other workgroups pass the caches, so scattered ones cost a memory
// request each: with most entries elsewhere (30,011 rows, random columns) an
// iteration took 30 us against 12 for the two kernels.  k_csr_rows therefore looks
// at the rows first: none longer than kCsrEntries, and no 256 rows with more than
// half of their entries in other pieces (a stencil's are at most the two
// outermost diagonals).  It runs ahead of the initialisation kernels, so the
// host's wait for its answer overlaps them; a solve that it sends to the kernels has
// paid 5 us.
//
// us per iteration, two kernels / here: 5-point FP64 4,225 rows 12.1 / 5.8, 65,025
// 12.4 / 7.9, FP32 11.7 / 4.5 and 12.1 / 5.6; 9 entries a row within 1,000 rows FP64,
// 30,011 rows 15.4 / 8.9.
#include "persist.hpp"

#include "persist_launch.hpp"
#include "tuning.hpp"

namespace pm
{
namespace
{

constexpr int kCsrEntries = 9;  // entries of a row at most (a 9-point stencil)

template <typename S, typename I>
struct CsrArgs
{
    int rows;
    const I* ro;
    const I* ci;
    const S* values;
    const S* x_in;
    S* x_out;
    S *p, *r, *s, *w, *u;
    const S* inv;
    const S* rhs;
    SolverState* st;
    double* region;
    PersistControl* ctl;
    word* xu;
    word* xx;
    unsigned tag;
    int count, per, leaders, refresh, t0, t_end, chunk, grow;
};

// *unfit = 1 (host memory) if a row is too long or most entries of the
// workgroup's rows lie outside their pieces of `piece` rows.
static_assert(kCsrEntries * kChunkRows <= kMaxWindows * kStreamCap, "rows the per-kernel SpMV walks lane by lane");
template <typename I>
__global__ __launch_bounds__(kBlock) void k_csr_rows(int64_t rows, const I* __restrict__ ro, const I* __restrict__ ci,
                                                     int piece, unsigned* unfit)
{
    __shared__ int sums[2][kBlock / kWave];
    const int64_t i = static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x;
    int entries = 0, away = 0;
    if (i < rows)
    {
        const int64_t b = static_cast<int64_t>(ro[i]), e = static_cast<int64_t>(ro[i + 1]);
        const int64_t first = i / piece * piece;
        if (e - b > kCsrEntries) *unfit = 1u;
        else
        {
            entries = static_cast<int>(e - b);
            for (int64_t k = b; k < e; ++k) away += static_cast<uint64_t>(ci[k] - first) >= static_cast<uint64_t>(piece);
        }
    }
    entries = wave_sum(entries);
    away = wave_sum(away);
    if (threadIdx.x % kWave == 0)
    {
        sums[0][threadIdx.x / kWave] = entries;
        sums[1][threadIdx.x / kWave] = away;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < kBlock / kWave; ++w)
    {
        sums[0][0] += sums[0][w];
        sums[1][0] += sums[1][w];
    }
    if (2 * sums[1][0] > sums[0][0]) *unfit = 1u;
}

template <typename S, typename I, bool JACOBI>
__global__ __launch_bounds__(kPersistThreads) void k_cg_csr(CsrArgs<S, I> a)
{
    using X = Exchange<S>;
    constexpr int NV = JACOBI ? 4 : 3;
    extern __shared__ char lds_raw[];
    S* us = reinterpret_cast<S*>(lds_raw);                      // u of the piece
    S* lv = us + kPersistThreads;                               // entries, [entry][lane]
    int* lc = reinterpret_cast<int*>(lv + kCsrEntries * kPersistThreads);  // a row of the piece, or ~(row of the matrix)
    double* red = reinterpret_cast<double*>(lc + kCsrEntries * kPersistThreads);
    __shared__ PersistShared<S> sh;

    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int blocks = gridDim.x, bid = blockIdx.x;
    const int g = static_cast<int>(xcd_logical_block(bid, blocks));
    const int rows = a.rows;
    const int piece = kPersistGroups * a.per * kChunkRows;  // per <= 4: at most a row per lane
    const int base = g * piece;
    int size = rows - base;
    size = size < 0 ? 0 : (size > piece ? piece : size);
    const int grp = tid / kBlock, gwave = wave % kWavesPerBlock;
    const int l = (grp * a.per + gwave) * kChunkRows + lane;
    const bool mine = gwave < a.per && l < size;
    const int i = mine ? base + l : 0;

    S p = mine ? a.p[i] : S(0), s = mine ? a.s[i] : S(0), x = mine ? a.x_in[i] : S(0);
    S r = mine ? a.r[i] : S(0), w = mine ? a.w[i] : S(0);
    const S inv = JACOBI && mine ? a.inv[i] : S(0);
    bool remote = false;  // some lane of the wavefront reads another piece
    {
        const int64_t b = mine ? static_cast<int64_t>(a.ro[i]) : 0;
        const int n = mine ? static_cast<int>(static_cast<int64_t>(a.ro[i + 1]) - b) : 0;
#pragma unroll
        for (int e = 0; e < kCsrEntries; ++e)
        {
            // an absent entry is 0 times the row's own u, which keeps the bits
            // of a finite sum
            lv[e * kPersistThreads + tid] = e < n ? a.values[b + e] : S(0);
            int c = mine ? l : 0;
            if (e < n)
            {
                const int full = static_cast<int>(a.ci[b + e]);
                c = full >= base && full < base + size ? full - base : ~full;
            }
            lc[e * kPersistThreads + tid] = c;
            remote = remote || c < 0;
        }
    }
    remote = __any(remote);
    us[tid] = S(0);
    const PersistWhere at{a.ctl, a.region, bid, blocks, g, a.count, a.leaders, a.t0, a.chunk, a.grow};
    if (tid == 0)
    {
        sh.hs.begin(a.st, a.t_end);
        sh.fail = given_up(&a.ctl->abort);
    }
    __syncthreads();
    auto u_of = [&]() { return JACOBI ? inv * r : r; };

    auto publish = [&](word* buf, unsigned tag, S v) {
        if (!mine) return;
        us[l] = v;
        X::put(buf, rows, i, v, tag);
    };
    // the lane's row of A v for the vector published last
    auto product = [&](const word* buf, unsigned tag, auto zero) {
        using Acc = decltype(zero);
        int c[kCsrEntries];
        word hw[kCsrEntries][X::kWords];
#pragma unroll
        for (int e = 0; e < kCsrEntries; ++e)
#pragma unroll
            for (int h = 0; h < X::kWords; ++h) hw[e][h] = 0;
        auto issue = [&]() {
#pragma unroll
            for (int e = 0; e < kCsrEntries; ++e)
                if (c[e] < 0) X::issue(buf, rows, ~c[e], hw[e]);
        };
        auto arrive = [&]() {
            auto arrived = [&]() {
                bool ok = true;
#pragma unroll
                for (int e = 0; e < kCsrEntries; ++e) ok = ok && (c[e] >= 0 || ready<S>(hw[e], tag));
                return ok;
            };
            return __all(arrived()) || wait_for(&a.ctl->abort, [&] {
                       issue();
                       return arrived();
                   });
        };
        auto gathered = [&](int e) {
            const S near = us[c[e] < 0 ? 0 : c[e]];
            return c[e] < 0 ? X::value(hw[e]) : near;
        };
#pragma unroll
        for (int e = 0; e < kCsrEntries; ++e) c[e] = lc[e * kPersistThreads + tid];
        bool fine = true;
        if (remote) issue();
        __syncthreads();
        Acc sum = zero;
        if (remote)
        {
            fine = arrive();
#pragma unroll
            for (int e = 0; e < kCsrEntries; ++e)
                sum = fma_s<Acc>(static_cast<Acc>(lv[e * kPersistThreads + tid]), static_cast<Acc>(gathered(e)), sum);
        }
        else
        {
#pragma unroll
            for (int e = 0; e < kCsrEntries; ++e)
                sum = fma_s<Acc>(static_cast<Acc>(lv[e * kPersistThreads + tid]), static_cast<Acc>(us[c[e]]), sum);
        }
        if (!fine) sh.fail = 1;
        return sum;
    };

    int code = kRunning;
    for (int t = a.t0;; ++t)
    {
        const unsigned tag = a.tag + static_cast<unsigned>(t - a.t0) + 1u;
        if (!persist_decide<S, NV>(sh, at, t, tag, red)) return;
        code = sh.code;
        if (code != kRunning) break;
        const S al = sh.alpha, be = sh.beta;
        const bool refresh = a.refresh > 0 && (t + 1) % a.refresh == 0;
        p = fma_s(be, p, u_of());
        s = fma_s(be, s, w);
        x = fma_s(al, p, x);
        if (!refresh) r = fma_s(-al, s, r);
        else
        {
            // r = b - A x with FP64 accumulation
            publish(a.xx, tag, x);
            const double ax = product(a.xx, tag, 0.0);
            if (mine) r = static_cast<S>(static_cast<double>(a.rhs[i]) - ax);
            __syncthreads();
        }
        publish(a.xu, tag, u_of());
        const S wn = product(a.xu, tag, S(0));
        w = mine ? wn : S(0);
        const double rv = static_cast<double>(r), uv = static_cast<double>(u_of());
        double part[kCgValues] = {0.0, 0.0, 0.0, 0.0};
        part[0] = __builtin_fma(rv, rv, 0.0);
        if (JACOBI) part[1] = __builtin_fma(rv, uv, 0.0);
        part[NV - 2] = __builtin_fma(static_cast<double>(w), uv, 0.0);
        part[NV - 1] = __builtin_fma(uv, static_cast<double>(s), 0.0);
        if (!persist_partials<S, NV>(sh, at, t, tag, part)) return;
    }

    const bool over = code == kHandOver;
    if (mine)
    {
        a.x_out[i] = x;
        if (over)
        {
            a.p[i] = p;
            a.s[i] = s;
            a.r[i] = r;
            a.w[i] = w;
            if (JACOBI) a.u[i] = u_of();
        }
    }
    if (over) persist_leave_partials<NV>(at);
    persist_end(sh, at, a.st, code);
}

// The split: a row per lane (the per-kernel workgroups hold at most four chunks
// of 64 rows), so up to 262,144 rows on 256 CUs.
static_assert(kPersistCsrRows == static_cast<int64_t>(kSolverGrid) * kBlock, "a row per lane of the solver grid");

int csr_per(const PersistProblem& p)
{
    return static_cast<int>(ceil_div(chunk_count(p.rows), static_cast<int64_t>(p.count)));
}

int csr_blocks(const PersistProblem& p) { return static_cast<int>(ceil_div(p.count, kPersistGroups)); }

template <typename S, typename I>
int csr_run(pm_workspace* ws, const PersistProblem& p, const I* ro, const I* ci, int64_t max_iterations,
            hipStream_t stream, int* outcome, int64_t* next, SolverState* state)
{
    CsrArgs<S, I> a{};
    a.rows = static_cast<int>(p.rows);
    a.ro = ro;
    a.ci = ci;
    a.values = static_cast<const S*>(p.a->values);
    a.x_in = static_cast<const S*>(p.x);
    a.x_out = static_cast<S*>(p.x_out);
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
    a.per = csr_per(p);
    const int blocks = csr_blocks(p);
    a.leaders = persist_leaders(blocks);
    a.refresh = p.refresh;
    a.chunk = p.chunk;
    a.grow = p.grow ? 1 : 0;
    const void* kernel = p.jacobi ? reinterpret_cast<const void*>(k_cg_csr<S, I, true>)
                                  : reinterpret_cast<const void*>(k_cg_csr<S, I, false>);
    const size_t lds = kPersistThreads * (sizeof(S) + kCsrEntries * (sizeof(S) + sizeof(int))) +
                       sizeof(double) * (p.count > kBlock ? (p.jacobi ? 4 : 3) * kRedEntries : 0);
    return persist_loop<S>(ws, p, a, kernel, blocks, lds, max_iterations, stream, outcome, next, state);
}

} // namespace

bool persist_csr_candidate(const PersistProblem& p, const pm_workspace* ws)
{
    return persist_enabled() && p.rows > 0 && p.rows <= kPersistCsrRows && p.a->nnz <= p.rows * kCsrEntries &&
           csr_per(p) <= kWavesPerBlock && persist_resident(ws, csr_blocks(p));
}

int persist_csr_look(pm_workspace* ws, const PersistProblem& p, hipStream_t stream)
{
    unsigned* unfit = &ws->host_state[1].counters[0];
    *unfit = 0u;
    const dim3 grid(static_cast<unsigned>(ceil_div(p.rows, kBlock)));
    const int piece = kPersistGroups * csr_per(p) * kChunkRows;
    if (use_compact(p.a))
        hipLaunchKernelGGL(k_csr_rows<int32_t>, grid, dim3(kBlock), 0, stream, p.rows, p.a->row_offsets32,
                           p.a->col_indices32, piece, unfit);
    else
        hipLaunchKernelGGL(k_csr_rows<int64_t>, grid, dim3(kBlock), 0, stream, p.rows, p.a->row_offsets,
                           p.a->col_indices, piece, unfit);
    PM_HIP(hipGetLastError());
    PM_HIP(hipEventRecord(ws->events[1], stream));
    return PM_OK;
}

int persist_csr_fits(pm_workspace* ws, bool* fits)
{
    PM_HIP(hipEventSynchronize(ws->events[1]));
    *fits = ws->host_state[1].counters[0] == 0u;
    return PM_OK;
}

int persist_csr_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                    int* outcome, int64_t* next, SolverState* state)
{
    const pm_csr* m = p.a;
    const bool compact = use_compact(m);
    if (p.dtype == PM_F64)
        return compact ? csr_run<double>(ws, p, m->row_offsets32, m->col_indices32, max_iterations, stream, outcome,
                                         next, state)
                       : csr_run<double>(ws, p, m->row_offsets, m->col_indices, max_iterations, stream, outcome, next,
                                         state);
    return compact ? csr_run<float>(ws, p, m->row_offsets32, m->col_indices32, max_iterations, stream, outcome, next,
                                    state)
                   : csr_run<float>(ws, p, m->row_offsets, m->col_indices, max_iterations, stream, outcome, next,
                                    state);
}

} // namespace pm
