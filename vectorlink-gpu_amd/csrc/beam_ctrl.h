// Device-side control block of one closest_vectors loop (ann.py:38-93).
// Batch-wide facts that the reference obtains with host round trips live here
// so that the per-iteration kernels can be enqueued back to back:
//   stop        - set once a checking iteration saw no row change (ann.py:90-91)
//   first[3]    - largest visited-list fill over all rows, one slot per iteration
//                 modulo 3 (iteration t reads t-1 and t, raises t+1, and rows of
//                 one launch may be in different phases); it is the first column
//                 that is empty in every row (utils.py:63-66) because rows are
//                 packed at the front (the fused step appends, the merge kernels
//                 keep them sorted as well)
//   changed[64] - ring of "some row changed" flags, one per checking iteration
//   sketch_rows - how many rows currently use the 8-bit sketch (they opt in once and may opt out once)
//   error       - a row found its own state impossible (see beam_row_state_ok)
// What the host needs to know at a progress check goes to a BeamReport in pinned host memory: the first workgroup of
// the launch after the checking iteration writes it (beam_gate) and the host, which has already enqueued that launch,
// polls it.  A copy of the flag and a wait for the stream instead left the GPU idle for 35 - 55 us per check (its five
// iterations of 256 queries at 4,096 x 128 take 105 us).
#pragma once
#include "vl_common.h"
#include "beam_report.h"

constexpr int kBeamStripes = 1024;

struct BeamCtrl {
    int stop;
    int ended_after;  // iterations run when stop was set (for callers that enqueue a fixed number of launches)
    int first[3];
    int changed[64];
    int sketch_rows;    // rows that currently look at their candidates through the 8-bit sketch first
    int error;          // set by a row whose visited-list fill is beyond what the iteration count allows: the
                        // workspace was overwritten while the loop ran (VL_ERR_STATE on the host)
    int refused_at;     // iteration that found the call's table of distances of no use (beam_table.hip), or 0
    int unordered;      // that table holds a distance that is not an ordinary number
    // profiling only, striped by workgroup so that the atomic adds do not queue up on one address:
    unsigned long long evals[kBeamStripes];   // candidate rows actually fetched
    unsigned long long wanted[kBeamStripes];  // candidate distances asked for (fetched or served by the cache)
    unsigned long long sketched[kBeamStripes];  // candidate rows looked at through the 8-bit sketch only
};

__device__ inline void beam_report(const BeamCtrl *c, int t, int R, BeamReport *out) {
    out->changed = c->changed[(t / R) & 63];
    out->sketch_rows = c->sketch_rows;
    out->error = c->error;
    if (c->refused_at) out->refused_at = c->refused_at;  // (0 when the call took the slot; each word is a trip to the host's memory)
    __hip_atomic_store(&out->check, t, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// A row's visited list holds at most Vt ids per earlier iteration and never more than its E slots.  A
// count beyond that was not written by this loop (its workspace is shared with another call): the row
// must not run - its copy loops would run to that count - and the loop ends with an error.
__device__ inline bool beam_row_state_ok(BeamCtrl *c, int cnt, int bound, bool writer) {
    const bool ok = cnt >= 0 && cnt <= bound;
    if (!ok && writer) {
        c->error = 1;
        c->stop = 1;
    }
    return __builtin_amdgcn_readfirstlane(ok) != 0;  // (in a scalar register, like what beam_gate returns)
}

// State of iteration t as seen by a kernel launched for it:
//   2  the loop has ended, do nothing
//   1  the visited list filled up earlier (add_new_to_seen_ returned None,
//      utils.py:68-69): the visit queue is no longer fed and pops yield empty ids
//   0  normal
// `writer` is true for exactly one thread of the launch, which records stop
// and clears the ring slot of the next checking iteration.
// look_at_fill = false (a launch that takes rows through several iterations, none of which can find a
// visited list full): state 1 is not looked for - rows of such a launch that finish early raise the slot of
// `first` that the launch after it reads, which for some lengths is the slot of iteration t - 1 modulo 3.
// report (may be null): where the launch after a checking iteration tells the host what that check found.
// The result is the same in all lanes of a workgroup, but by way of the writer's own branches the compiler takes it for
// one that lanes may disagree about, and with it everything that a kernel does after `if (gate) return`: barriers
// and loop ends inside a branch with a lane mask of its own, where it has reloaded spilled registers with no lane active.
// Hence the scalar register.
__device__ inline int beam_gate(BeamCtrl *c, int t, int R, int E, bool writer, BeamReport *report = nullptr,
                                bool look_at_fill = true) {
    int stop = c->stop;
    const bool after_check = t > 1 && ((t - 1) % R) == 0;
    if (writer && report && after_check) beam_report(c, t - 1, R, report);
    if (!stop && after_check && c->changed[((t - 1) / R) & 63] == 0) {
        stop = 1;
        if (writer) c->ended_after = t - 1;  // the loop ran t - 1 iterations
    }
    if (writer && stop) c->stop = 1;
    // the slot of the check after next: this iteration itself may be a checking one (R == 1)
    // and rows of one launch set their flag while others are still here
    if (writer && !stop && ((t - 1) % R) == 0) c->changed[((t - 1) / R + 2) & 63] = 0;
    const bool full = look_at_fill && t >= 2 && c->first[(t - 1) % 3] >= E;
    return __builtin_amdgcn_readfirstlane(stop ? 2 : full ? 1 : 0);
}
