// The resident form of the CG2D solve (mj_cg_resident.hip): eligibility, launch and its tables of a T plan.
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/mjamd.h"
#include "mj_internal.h"

namespace mj {
constexpr int kResMaxTiles = 16;  // tiles of a member (a wave polls two partial sums of each at once)

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
