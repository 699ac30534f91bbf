// Per-system state of a batched solve and the decision of its single-reduction
// form, shared by the per-kernel iteration (batch.hip) and the persistent one
// (persist_batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "spmv_kernels.hpp"
#include "workspace.hpp"

namespace pm
{

struct BatchState
{
    double rho;
    double alpha;
    double beta;
    double rr;
    double rr0;
    double tol;
    int32_t iteration;
    int32_t done;
    unsigned long long bad_row;
    double den;  // single-reduction form: p.Ap of the last direction

    // The decision after a completed step of the single-reduction form, from
    // r.r, gamma = r.u, delta = w.u and u.s: the stop code, else alpha and beta
    // of the next step.
    template <typename S>
    __device__ __forceinline__ int advance(double sum_rr, double gamma, double delta, double us,
                                           int32_t max_iterations)
    {
        int code = kRunning;
        // independent of the branches below, so that their latencies overlap
        const double root = sqrt(sum_rr), ratio = gamma / rho;
        double b = 0.0, d = delta, a = 0.0;
        iteration += 1;
        rr = sum_rr;
        if (!isfinite(sum_rr) || sum_rr < 0.0) code = kNonFinite;
        else if (root <= tol) code = kConverged;
        else if (iteration >= max_iterations) code = kIterationLimit;
        else
        {
            if (rho == 0.0 && gamma == 0.0) b = 0.0;
            else if (isfinite(rho) && isfinite(gamma) && rho > 0.0 && gamma > 0.0)
            {
                b = ratio;
                if (!isfinite(b) || !isfinite(static_cast<S>(b))) code = kBreakdown;
            }
            else code = kBreakdown;
            if (code == kRunning && b != 0.0) d = delta + b * (2.0 * us + b * den);
            if (code == kRunning && !(d > 0.0 && isfinite(d)))
            {
                b = 0.0;
                d = delta;
            }
        }
        if (code == kRunning && !step_length<S>(gamma, d, a)) code = kBreakdown;
        beta = b;
        alpha = a;
        rho = gamma;
        den = d;
        return code;
    }
};

} // namespace pm
