// Host-side helpers shared by the single-problem C ABI (hdg_api.hip) and the
// batches (hdg_batch.hip).  Not part of the public ABI.
#pragma once
#include "hdg_internal.h"

namespace hdg {

// Sizes of the vertex hierarchy of an nx x ny rectangle mesh: fills nlev,
// lev[1..nlev-1].nx, ny, n, npts and tail (no device arrays).
void mg_plan_levels(int nx, int ny, MgData& M);

}  // namespace hdg
