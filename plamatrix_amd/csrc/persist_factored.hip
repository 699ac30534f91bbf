// The persistent solve (persist.hip) with a factored preconditioner M^-1 = G^T G:
// A, G and G^T on the diagonal layout, G's diagonals the lower half of A's.
//
// Per iteration three products follow each other, t = G r, u = G^T t and w = A u,
// each of a vector that has just been formed, so r, t and u cross workgroups in
// turn and then the reduction: four exchange latencies instead of the two to four
// kernels of the per-kernel forms (112,320-row FP32 box: 13.3 us of kernels and two
// boundaries per iteration).  Vectors and the three matrices' values stay in
// registers.  Sums run in the order of the per-kernel forms, so a solve is bitwise
// theirs.
#include "persist.hpp"

#include <algorithm>
#include <type_traits>

#include "persist_launch.hpp"

namespace pm
{
namespace
{

template <typename S>
struct FactoredArgs
{
    int rows;
    DiaArgs dia, dia_g, dia_gt;
    const S *dv, *gv, *gtv;
    const uint16_t *mask, *gmask, *gtmask;
    const S* x_in;
    S* x_out;
    S *p, *r, *s, *w, *u;
    const S* rhs;
    SolverState* st;
    double* region;
    PersistControl* ctl;
    word* xu;  // exchange words: u, then x of a refresh, r, t
    word* xx;
    int words;  // of one vector
    unsigned tag;
    int count, per, halo, leaders, refresh, t0, t_end, chunk, grow;
    int window;  // bytes of an LDS window, then the leaders' reduction after three
};

template <typename S, int ND, int R, bool FAR>
__global__ __launch_bounds__(kPersistThreads) void k_cgf_persist(FactoredArgs<S> a)
{
    using X = Exchange<S>;
    constexpr int M = ND / 2;
    extern __shared__ char lds_raw[];
    __shared__ PersistShared<S> sh;

    const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const int blocks = gridDim.x, bid = blockIdx.x;
    const int g = static_cast<int>(xcd_logical_block(bid, blocks));
    const int rows = a.rows, H = a.halo;
    const int piece = kPersistGroups * a.per * kChunkRows;
    const int base = g * piece;
    int size = rows - base;
    size = size < 0 ? 0 : (size > piece ? piece : size);
    // the piece's r, t, u (and x in u's place during a refresh) with their halos
    S* win_r = reinterpret_cast<S*>(lds_raw) + H;
    S* win_t = reinterpret_cast<S*>(lds_raw + a.window) + H;
    S* win_u = reinterpret_cast<S*>(lds_raw + 2 * a.window) + H;
    double* red = reinterpret_cast<double*>(lds_raw + 3 * a.window);
    word* xr = a.xx + a.words;
    word* xt = xr + a.words;

    const int grp = tid / kBlock, gwave = wave % kWavesPerBlock;
    const int l0 = (grp * a.per + gwave) * kChunkRows + lane;
    const int slots = (a.per - gwave + kWavesPerBlock - 1) / kWavesPerBlock;
    const int limit = l0 + slots * kBlock < size ? l0 + slots * kBlock : size;

    // an absent entry has the value 0 and some finite partner
    S p[R], s[R], x[R], r[R], w[R], u[R], val[R][ND], gl[R][ND], gu[R][ND];
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = l0 + k * kBlock;
        const bool ok = l < limit;
        const int64_t i = ok ? base + l : 0;
        const unsigned m = ok ? a.mask[i] : 0u, mg = ok ? a.gmask[i] : 0u, mt = ok ? a.gtmask[i] : 0u;
        p[k] = ok ? a.p[i] : S(0);
        s[k] = ok ? a.s[i] : S(0);
        x[k] = ok ? a.x_in[i] : S(0);
        r[k] = ok ? a.r[i] : S(0);
        w[k] = ok ? a.w[i] : S(0);
        u[k] = ok ? a.u[i] : S(0);
#pragma unroll
        for (int d = 0; d < ND; ++d)
        {
            val[k][d] = ((m >> d) & 1u) ? dia_value(i, static_cast<int64_t>(rows), a.dia, a.dv, d) : S(0);
            if (d <= M)
                gl[k][d] = ((mg >> d) & 1u) ? dia_value(i, static_cast<int64_t>(rows), a.dia_g, a.gv, d) : S(0);
            if (d >= M)
                gu[k][d] = ((mt >> (d - M)) & 1u) ? dia_value(i, static_cast<int64_t>(rows), a.dia_gt, a.gtv, d - M)
                                                  : S(0);
        }
    }
    for (int l = tid; l < 3 * a.window / static_cast<int>(sizeof(S)); l += kPersistThreads)
        reinterpret_cast<S*>(lds_raw)[l] = S(0);
    const PersistWhere at{a.ctl, a.region, bid, blocks, g, a.count, a.leaders, a.t0, a.chunk, a.grow};
    if (tid == 0)
    {
        sh.hs.begin(a.st, a.t_end);
        sh.fail = given_up(&a.ctl->abort);
    }
    __syncthreads();

    auto publish = [&](word* buf, S* win, unsigned tag, const S (&v)[R]) {
        int l = l0;
        asm volatile("" : "+v"(l));
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const int lr = l + k * kBlock;
            if (lr >= limit) continue;
            win[lr] = v[k];
            if (FAR || lr < H || lr >= size - H) X::put(buf, rows, base + lr, v[k], tag);
        }
    };
    // acc[k] = sum over the diagonals D0 .. D1 of matrix value times the vector
    // published last, in increasing column order
    auto product = [&](auto d0, auto d1, const word* buf, const S* win, unsigned tag, const S (&own)[R],
                       const S (&mat)[R][ND], auto* acc) {
        using Acc = std::remove_reference_t<decltype(acc[0])>;
        constexpr int D0 = decltype(d0)::value, D1 = decltype(d1)::value;
        int l = l0;
        asm volatile("" : "+v"(l));
        word lo[R][X::kWords], hi[R][X::kWords];
        auto issue = [&]() {
#pragma unroll
            for (int k = 0; k < R; ++k)
            {
                const int i = base + l + k * kBlock;
                // every row is published under FAR: a clamped row's word arrives too
                if constexpr (D0 == 0)
                {
                    const int c = i + a.dia.off[0];
                    X::issue(buf, rows, c < 0 ? 0 : (c >= rows ? rows - 1 : c), lo[k]);
                }
                if constexpr (D1 == ND - 1)
                {
                    const int c = i + a.dia.off[ND - 1];
                    X::issue(buf, rows, c < 0 ? 0 : (c >= rows ? rows - 1 : c), hi[k]);
                }
            }
        };
        auto arrived = [&]() {
            bool ok = true;
#pragma unroll
            for (int k = 0; k < R; ++k)
            {
                if constexpr (D0 == 0) ok = ok && ready<S>(lo[k], tag);
                if constexpr (D1 == ND - 1) ok = ok && ready<S>(hi[k], tag);
            }
            return ok;
        };
        bool fine = true;
        if constexpr (FAR) issue();
        for (int h0 = 0; h0 < 2 * H; h0 += kPersistThreads)
        {
            const int h = h0 + tid;
            const int q = h < H ? h - H : size + (h - H);
            const int i = base + q;
            if (h >= 2 * H || size == 0 || i < 0 || i >= rows) continue;
            word hw[X::kWords];
            fine = wait_for(&a.ctl->abort, [&] {
                       X::issue(buf, rows, i, hw);
                       return ready<S>(hw, tag);
                   }) && fine;
            const_cast<S*>(win)[q] = X::value(hw);
        }
        __syncthreads();
        if constexpr (FAR)
        {
            if (!__all(arrived()))
                fine = wait_for(&a.ctl->abort, [&] {
                           issue();
                           return arrived();
                       }) && fine;
        }
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const int lr = l + k * kBlock;
            Acc sum = Acc(0);
#pragma unroll
            for (int d = D0; d <= D1; ++d)
            {
                S e;
                if (d == M) e = own[k];
                else if (FAR && d == 0) e = X::value(lo[k]);
                else if (FAR && d == ND - 1) e = X::value(hi[k]);
                else e = win[lr + a.dia.off[d]];
                sum = fma_s<Acc>(static_cast<Acc>(mat[k][d]), static_cast<Acc>(e), sum);
            }
            acc[k] = lr < limit ? sum : Acc(0);
        }
        if (!fine) sh.fail = 1;
    };
    using First = std::integral_constant<int, 0>;
    using Middle = std::integral_constant<int, M>;
    using Last = std::integral_constant<int, ND - 1>;

    int code = kRunning;
    for (int t = a.t0;; ++t)
    {
        const unsigned tag = a.tag + static_cast<unsigned>(t - a.t0) + 1u;
        if (!persist_decide<S, 4>(sh, at, t, tag, red)) return;
        code = sh.code;
        if (code != kRunning) break;
        const S al = sh.alpha, be = sh.beta;
        const bool refresh = a.refresh > 0 && (t + 1) % a.refresh == 0;
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            p[k] = fma_s(be, p[k], u[k]);
            s[k] = fma_s(be, s[k], w[k]);
            x[k] = fma_s(al, p[k], x[k]);
            if (!refresh) r[k] = fma_s(-al, s[k], r[k]);
        }
        if (refresh)
        {
            // r = b - A x with FP64 accumulation
            publish(a.xx, win_u, tag, x);
            double ax[R];
            product(First{}, Last{}, a.xx, win_u, tag, x, val, ax);
#pragma unroll
            for (int k = 0; k < R; ++k)
            {
                const int l = l0 + k * kBlock;
                if (l < limit) r[k] = static_cast<S>(static_cast<double>(a.rhs[base + l]) - ax[k]);
            }
        }
        S tr[R];
        publish(xr, win_r, tag, r);
        product(First{}, Middle{}, xr, win_r, tag, r, gl, tr);
        publish(xt, win_t, tag, tr);
        product(Middle{}, Last{}, xt, win_t, tag, tr, gu, u);
        publish(a.xu, win_u, tag, u);
        product(First{}, Last{}, a.xu, win_u, tag, u, val, w);

        double part[kCgValues] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < R; ++k)
        {
            const double rv = static_cast<double>(r[k]), uv = static_cast<double>(u[k]);
            part[0] = __builtin_fma(rv, rv, part[0]);
            part[1] = __builtin_fma(rv, uv, part[1]);
            part[2] = __builtin_fma(static_cast<double>(w[k]), uv, part[2]);
            part[3] = __builtin_fma(uv, static_cast<double>(s[k]), part[3]);
        }
        if (!persist_partials<S, 4>(sh, at, t, tag, part)) return;
    }

    const bool over = code == kHandOver;
#pragma unroll
    for (int k = 0; k < R; ++k)
    {
        const int l = l0 + k * kBlock;
        if (l >= limit) continue;
        const int i = base + l;
        a.x_out[i] = x[k];
        if (!over) continue;
        a.p[i] = p[k];
        a.s[i] = s[k];
        a.r[i] = r[k];
        a.w[i] = w[k];
        a.u[i] = u[k];
    }
    if (over) persist_leave_partials<4>(at);
    persist_end(sh, at, a.st, code);
}

struct FactoredShape
{
    int nd, rows_per_lane, per, blocks, halo, span;
    bool far;
    size_t window, lds;
};

bool factored_shape(const PersistProblem& p, FactoredShape* out)
{
    const DiaArgs &d = p.dia->args, &l = p.dia_g->args, &u = p.dia_gt->args;
    const int nd = d.ndiag;
    if (!p.dia->active || !p.dia_g->active || !p.dia_gt->active || (nd != 5 && nd != 7) || p.rows <= 0) return false;
    if (l.ndiag != nd / 2 + 1 || u.ndiag != nd / 2 + 1) return false;
    for (int k = 0; k < nd; ++k)
        if (d.off[k] != -d.off[nd - 1 - k]) return false;
    for (int k = 0; k <= nd / 2; ++k)
        if (l.off[k] != d.off[k] || u.off[k] != d.off[nd / 2 + k]) return false;
    FactoredShape s{};
    s.nd = nd;
    s.per = static_cast<int>(ceil_div(chunk_count(p.rows), static_cast<int64_t>(p.count)));
    const int need = (s.per + kWavesPerBlock - 1) / kWavesPerBlock;
    const int es = p.dtype == PM_F64 ? 8 : 4;
    // registers: six vectors and up to 15 matrix words per row
    if (need > (es == 4 ? 2 : 1)) return false;
    s.rows_per_lane = need;
    s.blocks = static_cast<int>(ceil_div(p.count, kPersistGroups));
    const int64_t piece = static_cast<int64_t>(kPersistGroups) * s.per * kChunkRows;
    s.span = std::max<int>(static_cast<int>(piece), ((kPersistGroups - 1) * s.per + kWavesPerBlock) * kChunkRows +
                                                        (s.rows_per_lane - 1) * kBlock);
    auto window = [&](int64_t halo) { return (static_cast<size_t>(s.span + 2 * halo) * es + 15) & ~size_t(15); };
    auto total = [&](int64_t halo) {
        return 3 * window(halo) + (p.count > kBlock ? sizeof(double) * 4 * kRedEntries : size_t(0));
    };
    int64_t halo = d.off[nd - 1];
    if (halo > piece || halo > kPersistThreads / 2 || total(halo) > kPersistLds)
    {
        halo = d.off[nd - 2];
        s.far = true;
        if (halo > piece || total(halo) > kPersistLds) return false;
    }
    s.halo = static_cast<int>(halo);
    s.window = window(halo);
    s.lds = total(halo);
    *out = s;
    return true;
}

template <typename S, int ND>
const void* factored_kernel(const FactoredShape& s)
{
    if (s.rows_per_lane == 1)
        return s.far ? reinterpret_cast<const void*>(k_cgf_persist<S, ND, 1, true>)
                     : reinterpret_cast<const void*>(k_cgf_persist<S, ND, 1, false>);
    if constexpr (sizeof(S) == 4)
        return s.far ? reinterpret_cast<const void*>(k_cgf_persist<S, ND, 2, true>)
                     : reinterpret_cast<const void*>(k_cgf_persist<S, ND, 2, false>);
    return nullptr;
}

template <typename S>
int factored_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream, int* outcome,
                 int64_t* next, SolverState* state)
{
    FactoredShape shape{};
    *outcome = kPersistAbandoned;
    if (!factored_shape(p, &shape)) return PM_OK;
    const void* kernel = shape.nd == 5 ? factored_kernel<S, 5>(shape) : factored_kernel<S, 7>(shape);
    if (kernel == nullptr) return PM_OK;
    FactoredArgs<S> a{};
    a.rows = static_cast<int>(p.rows);
    a.dia = p.dia->args;
    a.dia_g = p.dia_g->args;
    a.dia_gt = p.dia_gt->args;
    a.dv = static_cast<const S*>(p.dia->values);
    a.gv = static_cast<const S*>(p.dia_g->values);
    a.gtv = static_cast<const S*>(p.dia_gt->values);
    a.mask = p.dia->mask;
    a.gmask = p.dia_g->mask;
    a.gtmask = p.dia_gt->mask;
    a.x_in = static_cast<const S*>(p.x);
    a.x_out = static_cast<S*>(p.x_out);
    a.p = static_cast<S*>(p.p);
    a.r = static_cast<S*>(p.r);
    a.s = static_cast<S*>(p.s);
    a.w = static_cast<S*>(p.w);
    a.u = static_cast<S*>(p.u);
    a.rhs = static_cast<const S*>(p.rhs);
    a.st = p.st;
    a.region = p.region;
    a.words = a.rows * Exchange<S>::kWords;
    a.count = p.count;
    a.per = shape.per;
    a.halo = shape.halo;
    a.leaders = persist_leaders(shape.blocks);
    a.refresh = p.refresh;
    a.chunk = p.chunk;
    a.grow = p.grow ? 1 : 0;
    a.window = static_cast<int>(shape.window);
    return persist_loop<S>(ws, p, a, kernel, shape.blocks, shape.lds, max_iterations, stream, outcome, next, state, 4);
}

} // namespace

bool persist_factored_wanted(const PersistProblem& p, const pm_workspace* ws)
{
    FactoredShape s{};
    return persist_enabled() && factored_shape(p, &s) && persist_resident(ws, s.blocks);
}

int persist_factored_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                         int* outcome, int64_t* next, SolverState* state)
{
    if (p.dtype == PM_F64) return factored_run<double>(ws, p, max_iterations, stream, outcome, next, state);
    return factored_run<float>(ws, p, max_iterations, stream, outcome, next, state);
}

} // namespace pm
