// A whole single-reduction CG / Jacobi-PCG solve in one cooperative launch,
// for matrices on the diagonal layout.
//
// The per-kernel iteration streams every vector and the matrix through the
// caches once per iteration and pays a kernel boundary (64 Ki rows: 9.9 us per
// iteration, all latency; 2.1 M rows: 27.9 us for 113 MB).  Here a workgroup
// keeps its rows for the whole solve: p, s, x, r, w and the rows' matrix values
// live in registers (the chip's register files hold 128 MB), with a few words
// per row in LDS for the largest systems.  Those with 32 bytes of a vector per lane
// (eight FP32 rows, four FP64) do not fit the 128 registers of a lane: 20 to 170 spill,
// which bounds their iteration and still costs less than the kernels (below).  Per
// iteration only u crosses workgroups, and one reduction.
//
// Work split.  The per-kernel iteration sums its dot products in `count`
// workgroups of four wavefronts over contiguous 64-row chunks; a workgroup here
// takes four consecutive ones of those (1,024 threads), each wavefront the rows
// of the wavefront it stands for, and every sum runs in the same order.  A solve
// is therefore bitwise the per-kernel solve.
//
// Exchange.  Every word that crosses workgroups is a 64-bit relaxed atomic at
// agent scope that carries 32 bits of data and the iteration's tag, so a reader
// polls the data itself: no flags, fences or ordering between words.  (An
// agent-scope fence writes back or drops the XCD's L2: with fences a 65,536-row
// iteration took 27 us, with these words 5.)  A word is rewritten only after
// every reader of its old value has contributed to a reduction that the writer
// waited for; the partial sums, which several workgroups read, alternate
// between two sets.
//
// Rows near a workgroup's ends are copied into LDS halos; the outermost
// diagonals of a 3-D stencil reach whole pieces away, and their words are read
// by the lane that needs them.
//
// Waits are bounded: a workgroup that sees no progress for kWaitSeconds (or
// another one's notice of that) leaves, the new x is not committed, and the
// host runs the solve in the per-kernel form instead.
//
// Measured, solve time per-kernel / persistent: 65,536-row FP64 2-D Laplacian
// (767 iterations, one row per lane) 7.50 / 3.90 ms, 5.0 us per iteration, two
// exchange latencies; 2,097,152-row FP32 3-D diffusion (753 iterations, eight
// rows per lane) 21.2 / 15.2 ms with refinement, 18.6 us per iteration.
//
// us per iteration of 200-iteration solves, per-kernel / persistent, by diagonals and
// rows per lane (U: unit diagonal, J: Jacobi):
//   5 FP64 J   1: 262 k rows 21.3 / 8.3    2: 504 k 24.7 / 9.4    4: 1.04 M 34.2 / 12.7
//   7 FP64 U   1: 216 k 19.7 / 8.4         2: 493 k 23.1 / 12.4   4: not in LDS
//   7 FP64 J   1: 216 k 24.3 / 9.1         2: 493 k 28.5 / 13.5
//   5 FP32 J   2: 303 k 14.4 / 8.3         4: 1.0 M 20.8 / 9.9    8: 1.99 M 36.6 / 12.5
//   5 FP32 U   2: 303 k 11.8 / 7.3         4: 1.0 M 15.7 / 8.4    8: 1.99 M 27.4 / 10.3
//   7 FP32 J   2: 493 k 19.2 / 9.8         4: 1.0 M 26.1 / 12.1   8: 1.12 M 28.9 / 20.4, 2.1 M 38.2 / 21.9
//   7 FP32 U   2: 493 k 13.4 / 8.8         4: 1.0 M 17.7 / 10.7   8: 1.12 M 19.8 / 17.7, 2.1 M 28.0 / 20.9
// A launch costs more before its first iteration; solves of six iterations still gain up
// to four rows per lane (7 FP32 U 1.0 M: 356 / 327 us), with eight they are level (7 FP32
// U 384 / 386 us at 1.12 M rows, 463 / 490 at 2.0 M; J 699 / 650).
#include "persist.hpp"

#include <algorithm>
#include <type_traits>

#include "persist_launch.hpp"
#include "spmv_kernels.hpp"

namespace pm
{
namespace
{

template <typename S>
struct PersistArgs
{
    int rows;
    DiaArgs dia;
    const S* dv;
    const uint16_t* mask;
    const S* x_in;
    S* x_out;
    S *p, *r, *s, *w, *u;
    const S* inv;
    const S* rhs;
    SolverState* st;
    double* region;
    PersistControl* ctl;
    word* xu;  // u words: low halves (FP32: the value), then high halves
    word* xx;  // x words of a residual refresh
    unsigned tag;  // tags of this launch are above it
    int count, per, halo, leaders, refresh;
    int t0, t_end;
    int chunk, grow;
    int span;  // local rows that the LDS arrays hold
    int priv, red;  // bytes of LDS before x and the inner diagonals, and before the leaders' reduction
};

// ND diagonals with symmetric offsets (ND / 2 is the main diagonal), R rows per
// lane.  UNIT: an unpreconditioned solve whose main diagonal is all ones (u is
// r); else the main diagonal is stored and u = inv r (inv of ones without a
// preconditioner, which gives the same bits).  FAR: the outermost diagonals
// reach past the halos.  An absent entry has the value 0 and some finite
// partner, which leaves the row sums' bits alone.
//
// Registers: p, s, r, w, the two outermost diagonals (and inv, diagonal) per
// row, with x and the inner diagonals as long as a lane's rows stay below 32
// bytes per vector.  From there on x and the inner upper diagonals sit in LDS
// (a symmetric matrix: row l's lower value is row l - off's upper one).
template <typename S, int ND, int R, bool UNIT, bool FAR>
__global__ __launch_bounds__(kPersistThreads) void k_cg_persist(PersistArgs<S> a)
{
    using X = Exchange<S>;
    constexpr int M = ND / 2;
    constexpr bool kLds = sizeof(S) * R >= 32;
    constexpr int NV = UNIT ? 3 : 4;
    // far words in flight per lane: FB rows of two
    constexpr int FB = R < 8 / (2 * X::kWords) ? R : 8 / (2 * X::kWords);
    extern __shared__ char lds_raw[];
    __shared__ PersistShared<S> sh;

    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int blocks = gridDim.x, bid = blockIdx.x;
    const int g = static_cast<int>(xcd_logical_block(bid, blocks));
    const int rows = a.rows, H = a.halo;
    const int piece = kPersistGroups * a.per * kChunkRows;  // rows of a full piece
    const int base = g * piece;
    int size = rows - base;  // rows of this piece
    size = size < 0 ? 0 : (size > piece ? piece : size);
    S* us = reinterpret_cast<S*>(lds_raw) + H;         // u of rows [-H, span + H) of the piece
    S* xs = reinterpret_cast<S*>(lds_raw + a.priv);    // kLds: x, [R][kPersistThreads]
    S* vs = xs + R * kPersistThreads + H;              // kLds: inner upper diagonals of rows [-H, piece)
    const int vstride = a.span + H;
    double* red = reinterpret_cast<double*>(lds_raw + a.red);  // leaders: entries from kBlock on, [value][entry]

    // rows of the lane: local row l0 + k * kBlock for k < slots
    const int grp = tid / kBlock, gwave = wave % kWavesPerBlock;
    const int l0 = (grp * a.per + gwave) * kChunkRows + lane;
    const int slots = (a.per - gwave + kWavesPerBlock - 1) / kWavesPerBlock;
    const int limit = l0 + slots * kBlock < size ? l0 + slots * kBlock : size;  // local rows below it are the lane's

    S p[R], s[R], x[R], r[R], w[R], val[R][ND], inv[R];
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = l0 + k * kBlock;
        const bool ok = l < limit;
        const int i = ok ? base + l : 0;
        const unsigned m = ok ? a.mask[i] : 0u;
        p[k] = ok ? a.p[i] : S(0);
        s[k] = ok ? a.s[i] : S(0);
        r[k] = ok ? a.r[i] : S(0);
        w[k] = ok ? a.w[i] : S(0);
        if constexpr (!UNIT) inv[k] = ok ? (a.inv != nullptr ? a.inv[i] : S(1)) : S(0);
        const S xv = ok ? a.x_in[i] : S(0);
        if constexpr (kLds) xs[k * kPersistThreads + tid] = xv;
        else x[k] = xv;
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            if ((UNIT && d == M) || (kLds && d != 0 && d != M && d != ND - 1)) continue;
            val[k][d] = ((m >> d) & 1u)
                            ? dia_value(static_cast<int64_t>(i), static_cast<int64_t>(rows), a.dia, a.dv, d)
                            : S(0);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (kLds)
    {
#pragma unroll
        for (int d = M + 1; d < ND - 1; ++d)
            for (int l = tid - H; l < a.span; l += kPersistThreads)
            {
                const int i = base + l;
                vs[(d - M - 1) * vstride + l] =
                    i >= 0 && l < size && ((a.mask[i] >> d) & 1u) ? a.dv[static_cast<int64_t>(a.dia.slot[d]) * rows + i] : S(0);
            }
    }
    // halo rows past the matrix and the rows past a short piece stay 0
    for (int l = tid - H; l < a.span + H; l += kPersistThreads) us[l] = S(0);
    auto u_of = [&](int k) {
        if constexpr (UNIT) return r[k];
        else return inv[k] * r[k];
    };
    auto x_of = [&](int k) {
        if constexpr (kLds) return xs[k * kPersistThreads + tid];
        else return x[k];
    };

    const PersistWhere at{a.ctl, a.region, bid, blocks, g, a.count, a.leaders, a.t0, a.chunk, a.grow};
    if (tid == 0)
    {
        sh.hs.begin(a.st, a.t_end);
        sh.fail = given_up(&a.ctl->abort);
    }
    __syncthreads();

    // the lane's rows of a vector into LDS and, where another workgroup reads
    // them, into the exchange
    auto publish = [&](word* buf, unsigned tag, auto get) {
        int l = l0;
        asm volatile("" : "+v"(l));
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const int lr = l + k * kBlock;
            if (lr < limit)
            {
                const S v = get(k);
                us[lr] = v;
                if (FAR || lr < H || lr >= size - H) X::put(buf, rows, base + lr, v, tag);
            }
        }
    };

    // acc[k] = row k of A v for the vector published last, entries in
    // increasing column order; own(k) is the lane's own entry
    auto product = [&](const word* buf, unsigned tag, auto own, auto* acc) {
        using Acc = std::remove_reference_t<decltype(acc[0])>;
        int l = l0;
        asm volatile("" : "+v"(l));
        word far_lo[FB][X::kWords], far_hi[FB][X::kWords];
        // every row is published under FAR, so the word of a clamped row
        // (absent entries, slots past the lane's rows) arrives too
        auto issue = [&](int kb) {
#pragma unroll
            for (int j = 0; j < FB; ++j)
            {
                const int i = base + l + (kb + j) * kBlock;
                int lo = i + a.dia.off[0], hi = i + a.dia.off[ND - 1];
                lo = lo < 0 ? 0 : (lo >= rows ? rows - 1 : lo);
                hi = hi < 0 ? 0 : (hi >= rows ? rows - 1 : hi);
                X::issue(buf, rows, lo, far_lo[j]);
                X::issue(buf, rows, hi, far_hi[j]);
            }
        };
        auto arrived = [&]() {
            bool ok = true;
#pragma unroll
            for (int j = 0; j < FB; ++j) ok = ok && ready<S>(far_lo[j], tag) && ready<S>(far_hi[j], tag);
            return ok;
        };
        bool fine = true;
        if constexpr (FAR) issue(0);
        // halo rows of the neighbouring pieces
        for (int h0 = 0; h0 < 2 * H; h0 += kPersistThreads)
        {
            const int h = h0 + tid;
            const int q = h < H ? h - H : size + (h - H);
            const int i = base + q;
            if (h >= 2 * H || size == 0 || i < 0 || i >= rows) continue;
            word hw[X::kWords];
            fine = fine && wait_for(&a.ctl->abort, [&] {
                       X::issue(buf, rows, i, hw);
                       return ready<S>(hw, tag);
                   });
            us[q] = X::value(hw);
        }
        __syncthreads();
#pragma unroll
        for (int kb = 0; kb < R; kb += FB)
        {
            if constexpr (FAR)
            {
                if (!__all(arrived()))
                    fine = fine && wait_for(&a.ctl->abort, [&] {
                               issue(kb);
                               return arrived();
                           });
            }
#pragma unroll
            for (int j = 0; j < FB; ++j)
            {
                const int k = kb + j;
                // slots past the lane's rows compute on whatever the LDS behind
                // the piece holds and are dropped
                const int lr = l + k * kBlock;
                Acc sum = Acc(0);
#pragma unroll
                for (int d = 0; d < ND; ++d)
                {
                    S v, e;
                    if (d == M) e = own(k);
                    else if (FAR && (d == 0 || d == ND - 1)) e = X::value(d == 0 ? far_lo[j] : far_hi[j]);
                    else e = us[lr + a.dia.off[d]];
                    if (d == M)
                    {
                        if constexpr (UNIT) v = S(1);
                        else v = val[k][d];
                    }
                    else if (!kLds || d == 0 || d == ND - 1) v = val[k][d];
                    else if (d < M) v = vs[(ND - 1 - d - M - 1) * vstride + lr + a.dia.off[d]];
                    else v = vs[(d - M - 1) * vstride + lr];
                    sum = fma_s<Acc>(static_cast<Acc>(v), static_cast<Acc>(e), sum);
                }
                acc[k] = l + k * kBlock < limit ? sum : Acc(0);
                if (kLds) __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (FAR)
                if (kb + FB < R) issue(kb + FB);
        }
        if (!fine) sh.fail = 1;
    };

    int code = kRunning;
    for (int t = a.t0;; ++t)
    {
        // ---- decision: stop test, alpha, beta from the partials of t - 1 ----
        const unsigned tag = a.tag + static_cast<unsigned>(t - a.t0) + 1u;
        if (!persist_decide<S, NV>(sh, at, t, tag, red)) return;
        code = sh.code;
        if (code != kRunning) break;
        const S al = sh.alpha, be = sh.beta;

        // ---- step, then w = A u of the new u ----
        const bool refresh = a.refresh > 0 && (t + 1) % a.refresh == 0;
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            p[k] = fma_s(be, p[k], u_of(k));
            s[k] = fma_s(be, s[k], w[k]);
            const S xn = fma_s(al, p[k], x_of(k));
            if constexpr (kLds) xs[k * kPersistThreads + tid] = xn;
            else x[k] = xn;
            if (!refresh) r[k] = fma_s(-al, s[k], r[k]);
        }
        if (refresh)
        {
            // r = b - A x with FP64 accumulation
            publish(a.xx, tag, x_of);
            double ax[R];
            product(a.xx, tag, x_of, ax);
#pragma unroll
            for (int k = 0; k < R; ++k)
            {
                const int l = l0 + k * kBlock;
                if (l < limit) r[k] = static_cast<S>(static_cast<double>(a.rhs[base + l]) - ax[k]);
            }
            __syncthreads();
        }
        publish(a.xu, tag, u_of);
        product(a.xu, tag, u_of, w);

        // ---- partial sums per workgroup of the per-kernel iteration ----
        double part[kCgValues] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const double rv = static_cast<double>(r[k]);
            const double uv = static_cast<double>(u_of(k));
            part[0] = __builtin_fma(rv, rv, part[0]);
            if (!UNIT) part[1] = __builtin_fma(rv, uv, part[1]);
            part[NV - 2] = __builtin_fma(static_cast<double>(w[k]), uv, part[NV - 2]);
            part[NV - 1] = __builtin_fma(uv, static_cast<double>(s[k]), part[NV - 1]);
        }
        if (!persist_partials<S, NV>(sh, at, t, tag, part)) return;
    }

    // ---- the end: x, and for a hand-over everything the next form reads ----
    const bool over = code == kHandOver;
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = l0 + k * kBlock;
        if (l >= limit) continue;
        const int i = base + l;
        a.x_out[i] = x_of(k);
        if (!over) continue;
        a.p[i] = p[k];
        a.s[i] = s[k];
        a.r[i] = r[k];
        a.w[i] = w[k];
        if (!UNIT && a.inv != nullptr) a.u[i] = u_of(k);
    }
    if (over) persist_leave_partials<NV>(at);
    persist_end(sh, at, a.st, code);
}

struct PersistShape
{
    int nd, rows_per_lane, per, blocks, halo, span;
    bool unit, far;
    size_t shared, red;  // LDS before x and the inner diagonals, before the leaders' reduction
    size_t lds;
};

bool persist_shape(const PersistProblem& p, PersistShape* out)
{
    const DiaLayout& d = *p.dia;
    const int nd = d.args.ndiag;
    if (!d.active || (nd != 5 && nd != 7) || p.rows <= 0) return false;
    for (int k = 0; k < nd; ++k)
        if (d.args.off[k] != -d.args.off[nd - 1 - k]) return false;
    PersistShape s{};
    s.nd = nd;
    s.unit = !p.jacobi && d.args.slot[nd / 2] < 0;
    const int64_t chunks = chunk_count(p.rows);
    s.per = static_cast<int>(ceil_div(chunks, static_cast<int64_t>(p.count)));
    const int need = (s.per + kWavesPerBlock - 1) / kWavesPerBlock;
    s.rows_per_lane = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 8;
    const int es = p.dtype == PM_F64 ? 8 : 4;
    if (need > 8 || s.rows_per_lane * es > 32) return false;
    const bool in_lds = s.rows_per_lane * es == 32;  // x and the inner upper diagonals in LDS
    for (int k = 0; in_lds && k < nd / 2; ++k)
        if (d.args.slot[k] != d.args.slot[nd - 1 - k] || d.args.slot[k] < 0) return false;  // not mirrored
    s.blocks = static_cast<int>(ceil_div(static_cast<int64_t>(p.count), static_cast<int64_t>(kPersistGroups)));
    const int64_t piece = static_cast<int64_t>(kPersistGroups) * s.per * kChunkRows;
    const int inner_arrays = nd / 2 - 1;
    // the last local row any lane's R slots address
    s.span = ((kPersistGroups - 1) * s.per + kWavesPerBlock) * kChunkRows + (s.rows_per_lane - 1) * kBlock;
    s.span = std::max(s.span, static_cast<int>(piece));
    // the piece's u with its halos, x and the inner upper diagonals, and the
    // leaders' reduction of more than kBlock partials
    auto shared = [&](int64_t halo) { return (static_cast<size_t>(s.span + 2 * halo) * es + 15) & ~size_t(15); };
    auto reduction = [&](int64_t halo) {
        const size_t kept = in_lds ? (static_cast<size_t>(s.rows_per_lane) * kPersistThreads +
                                      static_cast<size_t>(inner_arrays) * (s.span + halo)) *
                                         es
                                   : 0;
        return (shared(halo) + kept + 15) & ~size_t(15);
    };
    auto total = [&](int64_t halo) {
        return reduction(halo) + (p.count > kBlock ? sizeof(double) * (s.unit ? 3 : 4) * kRedEntries : size_t(0));
    };
    // halos of the widest offset that a piece and the LDS can hold; only the
    // outermost diagonals may reach past it
    const int64_t outer = d.args.off[nd - 1], inner = d.args.off[nd - 2];
    int64_t halo = outer;
    if (halo > piece || halo > 2 * kPersistThreads || total(halo) > kPersistLds)
    {
        halo = inner;
        s.far = true;
        if (halo > piece || total(halo) > kPersistLds) return false;
    }
    s.halo = static_cast<int>(halo);
    s.shared = shared(halo);
    s.red = reduction(halo);
    s.lds = total(halo);
    *out = s;
    return true;
}

template <typename S, int ND, int R>
const void* persist_instance(const PersistShape& s)
{
    if (s.unit)
        return s.far ? reinterpret_cast<const void*>(k_cg_persist<S, ND, R, true, true>)
                     : reinterpret_cast<const void*>(k_cg_persist<S, ND, R, true, false>);
    return s.far ? reinterpret_cast<const void*>(k_cg_persist<S, ND, R, false, true>)
                 : reinterpret_cast<const void*>(k_cg_persist<S, ND, R, false, false>);
}

template <typename S, int ND>
const void* persist_kernel(const PersistShape& s)
{
    switch (s.rows_per_lane)
    {
    case 1: return persist_instance<S, ND, 1>(s);
    case 2: return persist_instance<S, ND, 2>(s);
    case 4: return persist_instance<S, ND, 4>(s);
    default: break;
    }
    if constexpr (sizeof(S) == 4) return persist_instance<S, ND, 8>(s);
    return nullptr;
}

template <typename S>
int persist_run_t(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream, int* outcome,
                  int64_t* next, SolverState* state)
{
    PersistShape shape{};
    *outcome = kPersistAbandoned;
    if (!persist_shape(p, &shape)) return PM_OK;
    const void* kernel = shape.nd == 5 ? persist_kernel<S, 5>(shape) : persist_kernel<S, 7>(shape);
    if (kernel == nullptr) return PM_OK;
    PersistArgs<S> a{};
    a.rows = static_cast<int>(p.rows);
    a.dia = p.dia->args;
    a.dv = static_cast<const S*>(p.dia->values);
    a.mask = p.dia->mask;
    a.x_in = static_cast<const S*>(p.x);
    a.x_out = static_cast<S*>(p.x_out);
    a.p = static_cast<S*>(p.p);
    a.r = static_cast<S*>(p.r);
    a.s = static_cast<S*>(p.s);
    a.w = static_cast<S*>(p.w);
    a.u = static_cast<S*>(p.u);
    a.inv = p.jacobi ? static_cast<const S*>(p.inv) : nullptr;
    a.rhs = static_cast<const S*>(p.rhs);
    a.st = p.st;
    a.region = p.region;
    a.count = p.count;
    a.per = shape.per;
    a.halo = shape.halo;
    a.priv = static_cast<int>(shape.shared);
    a.red = static_cast<int>(shape.red);
    a.span = shape.span;
    a.leaders = persist_leaders(shape.blocks);
    a.refresh = p.refresh;
    a.chunk = p.chunk;
    a.grow = p.grow ? 1 : 0;
    return persist_loop<S>(ws, p, a, kernel, shape.blocks, shape.lds, max_iterations, stream, outcome, next, state);
}

} // namespace

bool persist_wanted(const PersistProblem& p, const pm_workspace* ws)
{
    PersistShape s{};
    return persist_enabled() && persist_shape(p, &s) && persist_resident(ws, s.blocks);
}

int persist_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream, int* outcome,
                int64_t* next, SolverState* state)
{
    if (p.dtype == PM_F64) return persist_run_t<double>(ws, p, max_iterations, stream, outcome, next, state);
    return persist_run_t<float>(ws, p, max_iterations, stream, outcome, next, state);
}

} // namespace pm
