// Persistent solve of a batch's short-row systems (persist_batch.hip).
#pragma once

#include <vector>

#include "batch_state.hpp"

namespace pm
{

// What the device saw of one system's rows.
struct BatchLook
{
    int band;  // largest |column - row|, or the largest int: not for a team
};

// A batched CG / Jacobi solve after its initialisation: r, w (q), p (p0),
// s (p1) and the states of iteration 0 are in place.
struct BatchTeams
{
    const pm_csr* a;
    int64_t systems;
    const int64_t* begin;      // host: first row of every system
    const int64_t* end;        // host: one past its last
    const uint8_t* skip;       // host: systems that another preconditioner or form takes
    const int32_t* chunk_sys;  // device
    int64_t chunks;
    const int64_t* sys_end;    // device
    const int64_t* sys_chunk0; // device: first 64-row chunk
    const void* rhs;
    void* x;
    const void *r, *w, *p, *s;
    const void* inv;           // null: no preconditioner
    void* x_out;               // scratch vector
    BatchState* st;
    unsigned long long* done_count;
    int32_t max_iterations;
    int refresh;
};

// Looks at the rows of every system of a fitting size (once per matrix and call) into
// `look`; waits for the stream if there is one.
int batch_teams_look(pm_workspace* ws, const BatchTeams& b, std::vector<BatchLook>& look, hipStream_t stream);
// Solves every system that fits, committing x, its state and the stopped
// count; the others are left as they are.  *ran: there was one.  Waits for the stream.
int batch_teams_run(pm_workspace* ws, const BatchTeams& b, const std::vector<BatchLook>& look, hipStream_t stream,
                    bool* ran);

} // namespace pm
