// What a launch that runs many single-reduction iterations keeps between its
// decisions (persist.hip, persist_small.hip).
#pragma once

#include "cg_rules.hpp"
#include "persist.hpp"

namespace pm
{

constexpr int kHandOver = 100;      // decision code: leave without deciding
constexpr int kCounterOutcome = 1;  // SolverState::counters slot: what became of a launch
constexpr int kCounterNext = 2;     // ... iteration the launch handed over at
constexpr int kCounterOver = 3;     // ... iteration a restart hands over at (0: none yet)

// Kept in LDS by the one thread that decides: as registers it would take some
// from every lane.
struct PersistHistory
{
    CgHistory h;
    double rr, rr0, alpha;
    int completed, t_stop;
    int over;  // iteration a restart hands over at, in this launch or a later one; 0: none

    // before iteration t0 (even) of a solve, launched up to iteration t_end
    __device__ __forceinline__ void begin(const SolverState* st, int t_end)
    {
        h = CgHistory{st->max_iterations, st->tol_rule, st->rel_tol, st->abs_tol,
                      st->tol,            st->rho[1],   st->den[1],  st->bad_row != ~0ull};
        completed = st->iter[1] + 1;
        rr0 = st->rr0;
        rr = alpha = 0.0;
        over = static_cast<int>(st->counters[kCounterOver]);
        t_stop = over != 0 && over < t_end ? over : t_end;
    }

    // The decision at the head of iteration t; kHandOver at the iteration the
    // launch ends at.
    template <typename S>
    __device__ __forceinline__ int decide(int t, double sum_rr, double gamma, double delta, double us, int chunk,
                                          bool grow, S& step, S& beta)
    {
        if (t >= t_stop) return kHandOver;
        const CgDecision d = cg_rules<S>(h, completed, sum_rr, gamma, delta, us);
        step = static_cast<S>(d.alpha);
        beta = static_cast<S>(d.beta);
        rr = sum_rr;
        alpha = d.alpha;
        if (completed == 0) rr0 = sum_rr;
        h.tol = d.tol;
        h.gamma_prev = gamma;
        h.den_prev = d.den;
        // one thread decides while the others wait: the rare branch out of its way (0.2 %
        // of a 767-iteration solve)
        if (__builtin_expect(d.restart, 0) && over == 0)
        {
            const int64_t at = hand_over_iteration(t, chunk, grow, kMaxGrownChunk);
            over = at < INT32_MAX ? static_cast<int>(at) : INT32_MAX;
            if (over < t_stop) t_stop = over;
        }
        ++completed;
        return d.code;
    }

    // The state record as the per-kernel iteration would have left it.
    __device__ __forceinline__ void record(SolverState* st, int code) const
    {
        // completed counts the decisions: the last one saw completed - 1 updates
        const int seen = completed - 1, par = seen & 1;
        st->rr = rr;
        st->rr0 = rr0;
        st->tol = h.tol;
        st->iteration = seen;
        st->iter[par] = seen;
        st->rho[par] = h.gamma_prev;
        st->den[par] = h.den_prev;
        st->alpha = alpha;
        st->counters[kCounterOver] = static_cast<unsigned>(over);
        if (over != 0 && (code != kHandOver || completed >= over)) st->counters[kCounterRestart] = 1u;
        st->counters[kCounterNext] = static_cast<unsigned>(completed);
        if (code != kHandOver) st->done = code;
    }
};

} // namespace pm
