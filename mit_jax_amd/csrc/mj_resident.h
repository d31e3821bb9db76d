// The resident form of the CG2D solve (mj_cg_resident.hip): eligibility, launch and its tables of a T plan.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "../../include/mjamd.h"
#include "mj_internal.h"

namespace mj {
constexpr int kResMaxTiles = 16;  // tiles of a member (a wave polls two partial sums of each at once)

// What the workgroups of a resident solve share, in the workspace. A group is one workgroup per tile of a member.
struct ResSync {
    uint64_t* words;     // per group: [2][nslots][2] ring values, [2][T][4] partial sums, by parity of the exchange
    size_t group_words;
    uint64_t* next;      // [G] the group's current member
    int* queue;          // members taken so far
    int* error;          // a wait timed out
    unsigned long long limit;  // ticks a wait may take; it looks at the clock every 1024 polls, 0: at every one
    const int* order;    // [B] the order in which members are taken, or NULL (as they come)
    int G, T, nslots, B;
};
// Fills y for a cooperative launch of kfn (threads, dynamic LDS) over cfg's batch and clears its words on the stream;
// *ok false (and nothing enqueued) when the device or the workspace does not allow it.
int resident_prepare(const mj_halo_plan* P, const mj_cg2d_ops* ops, const mj_cg2d_config* cfg, const void* kfn,
                     int threads, size_t lds, void* workspace, size_t workspace_bytes, hipStream_t st, ResSync* y,
                     bool* ok);
// The launch of kfn (y.G * y.T blocks); diag's records say -2 if a wait in it failed.
int resident_launch(const void* kfn, int threads, void** args, size_t lds, const ResSync& y, mj_cg2d_diag* diag,
                    hipStream_t st);
// Whether a stream is being captured into a graph (the resident launches are not for that).
int stream_capturing(hipStream_t st, bool* capturing);

// Whether the solve of this configuration can run resident (layout and plan).
bool resident_fits(const mj_halo_plan* P, const mj_cg2d_config* c);
// Launches the solve; *done false (and nothing launched) when the device or the workspace does not allow it.
int resident_solve(mj_halo_plan* P, const mj_cg2d_ops* ops, const double* b, const double* x0, double* x,
                   const double* cg2dNorm, const mj_cg2d_config* cfg, void* workspace, size_t workspace_bytes,
                   mj_cg2d_diag* diag, hipStream_t st, bool* done);
// Part of ensure_cg_tables: the resident tables of a plan whose tiles are 90 x 90 (others: left without).
int ensure_resident_tables(mj_halo_plan* P, const std::vector<int32_t>& roff, const std::vector<int32_t>& rdst,
                           const std::vector<int32_t>& rsrc, const std::vector<int8_t>& rsg);
}  // namespace mj
