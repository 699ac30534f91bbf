// Persistent single-reduction CG / Jacobi-PCG: one launch runs a whole solve,
// cooperative on the diagonal layout (persist.hip) and on CSR matrices of short
// rows (persist_csr.hip), in one workgroup on small CSR matrices
// (persist_small.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dia.hpp"
#include "workspace.hpp"

namespace pm
{

// Rows that the persistent solve of a CSR matrix takes, at most: a row per lane.
constexpr int64_t kPersistCsrRows = 262144;

// Largest chunk of iterations a solve's schedule grows to (adaptive_solve).
constexpr int kMaxGrownChunk = 64;

// A solve whose vectors sit where the per-kernel iteration keeps them between
// chunks: r, u (z; with a preconditioner), w (q), p (p0) and s (p1), the partials
// of the initialisation in region 1.
struct PersistProblem
{
    int64_t rows;
    int32_t dtype;
    const pm_csr* a;
    const DiaLayout *dia, *dia_g, *dia_gt;
    bool jacobi;
    const void* rhs;
    void* x;
    void *r, *u, *w, *p, *s;
    const void* inv;
    void* x_out;       // scratch vector the new x is written to before it is committed to x (null where no form needs it)
    SolverState* st;
    double* region;    // partials of iteration t0 - 1 (t0 even)
    int count;         // workgroups of the per-kernel iteration (its partial sums)
    int refresh;       // residual refresh interval, 0: never
    int chunk;         // the host's chunk schedule: first chunk, and whether chunks grow
    bool grow;
};

enum PersistOutcome : int
{
    kPersistStopped = 1,   // the state record holds the end of the solve
    kPersistHandOver = 2,  // after a restart: continue at iteration *next in the three-kernel form
    kPersistAbandoned = 3, // nothing was committed: x is as before, start again in another form
};

// Whether the persistent iteration on the diagonal layout takes this solve.
bool persist_wanted(const PersistProblem& p, const pm_workspace* ws);

// Runs the solve and waits for it.  *state receives the final state record.
int persist_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream, int* outcome,
                int64_t* next, SolverState* state);

// The same for the one-workgroup solve of a small CSR matrix.
bool persist_small_wanted(const PersistProblem& p);
int persist_small_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                      int* outcome, int64_t* next, SolverState* state);

// The same for CSR matrices of short, mostly local rows: a candidate by its
// sizes, the device's look at its rows (stream-ordered) and the answer (waits for
// the look only).
bool persist_csr_candidate(const PersistProblem& p, const pm_workspace* ws);
int persist_csr_look(pm_workspace* ws, const PersistProblem& p, hipStream_t stream);
int persist_csr_fits(pm_workspace* ws, bool* fits);
int persist_csr_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                    int* outcome, int64_t* next, SolverState* state);

// The same with a factored preconditioner, all three matrices on the diagonal
// layout (persist_factored.hip).
bool persist_factored_wanted(const PersistProblem& p, const pm_workspace* ws);
int persist_factored_run(pm_workspace* ws, const PersistProblem& p, int64_t max_iterations, hipStream_t stream,
                         int* outcome, int64_t* next, SolverState* state);

// The chunk schedule of an adaptive solve: chunk c covers iterations
// [end(c - 1), end(c)).  Both forms of a solve must leave the single-reduction
// form at the same iteration after a restart.
__host__ __device__ inline int64_t next_chunk(int64_t issued, int64_t size, bool grow, int64_t most)
{
    return grow && issued >= 2 && size < most ? size * 2 : size;
}

// The iteration a restart at iteration t hands over at: the chunk that holds t
// and the one after it are already in flight when the host reads the flag.
__host__ __device__ inline int64_t hand_over_iteration(int64_t t, int64_t first, bool grow, int64_t most)
{
    int64_t end = 0, size = first, issued = 0;
    do
    {
        end += size;
        size = next_chunk(++issued, size, grow, most);
    } while (end <= t);
    return end + size;
}

} // namespace pm
