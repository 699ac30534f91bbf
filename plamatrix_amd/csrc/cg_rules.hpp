// The stop test and step rules of one single-reduction CG / PCG iteration,
// shared by the per-kernel iteration (pcg.hip) and the persistent one
// (persist.hip), so that both decide alike from the same reduced values.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "spmv_kernels.hpp"
#include "workspace.hpp"

namespace pm
{

constexpr int kCounterRestart = 0;  // SolverState::counters slot: a single-reduction restart happened
constexpr int kCgValues = 4;        // r.r, r.u, w.u, u.s

// What the decision at the head of an iteration needs besides the reduced
// values: the solve's limits and the previous iteration's gamma and den.
struct CgHistory
{
    int32_t max_iterations;
    int32_t tol_rule;
    double rel_tol, abs_tol;
    double tol;         // valid once an iteration has completed
    double gamma_prev;  // ... likewise
    double den_prev;
    bool bad_diagonal;
};

struct CgDecision
{
    int code;  // Done
    bool restart;
    double tol, alpha, beta, den;
};

template <typename S>
__device__ __forceinline__ CgDecision cg_rules(const CgHistory& h, int completed, double rr, double gamma,
                                               double delta, double us)
{
    CgDecision d;
    d.restart = false;
    // independent of each other and of the branches below, so that their
    // latencies overlap: this runs in one thread while the others wait
    const double root = sqrt(rr);
    const double ratio = gamma / h.gamma_prev;
    // the accelerated solvers' max(abs, rel ||r0||), or the reference CPU
    // Schur solver's abs + rel ||r0|| (block_schur_cpu_solver.h:34-35)
    d.tol = completed != 0 ? h.tol
            : h.tol_rule   ? h.abs_tol + h.rel_tol * root
                           : fmax(h.abs_tol, h.rel_tol * root);
    d.code = kRunning;
    d.beta = 0.0;
    d.alpha = 0.0;
    d.den = delta;
    if (!isfinite(rr) || rr < 0.0) d.code = completed == 0 ? kInitNonFinite : kNonFinite;
    else if (root <= d.tol) d.code = kConverged;
    else if (completed == 0 && h.bad_diagonal) d.code = kBadDiagonal;
    else if (completed >= h.max_iterations) d.code = kIterationLimit;
    else
    {
        if (completed > 0)
        {
            // betaKernel, iterative_solver_kernels.cuh:204-238
            if (h.gamma_prev == 0.0 && gamma == 0.0) d.beta = 0.0;
            else if (isfinite(h.gamma_prev) && isfinite(gamma) && h.gamma_prev > 0.0 && gamma > 0.0)
            {
                d.beta = ratio;
                if (!isfinite(d.beta) || !isfinite(static_cast<S>(d.beta))) d.code = kBreakdown;
            }
            else d.code = kBreakdown;
            // u.s exists only after a completed step
            if (d.code == kRunning && d.beta != 0.0) d.den = delta + d.beta * (2.0 * us + d.beta * h.den_prev);
            // a non-positive p.Ap of the new direction restarts the step from
            // u (beta = 0, p.Ap = u.Au = delta); only a non-positive delta is
            // a breakdown of A itself
            if (d.code == kRunning && !(d.den > 0.0 && isfinite(d.den)))
            {
                d.beta = 0.0;
                d.den = delta;
                d.restart = true;
            }
        }
        if (d.code == kRunning && !step_length<S>(gamma, d.den, d.alpha)) d.code = kBreakdown;
    }
    return d;
}

} // namespace pm
