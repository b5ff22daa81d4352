// mdmc_adjoint.h -- launchers of the adjoint passes (mdmc_adjoint.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mdmc_internal.h"

namespace mdmc {

// per dual vertex: 8 corner contributions (contrib[8V]) from dL/dpos (dpos[3V]); clears
// clear[0, nClear) in the same launch (clear null: nothing)
void launchAdjointVertex(const GridDev& g, float iso, const int32_t* adjMap, const int32_t* adjCell, int64_t V, const float* dpos, float* contrib,
                         float* clear, int64_t nClear, hipStream_t s);
// dL/dvalue of the points near the surface of the grid inDims, whose processed grid outDims is
// itself (pad 0, outDims = inDims) or itself padded by one (pad 1): out is cleared beforehand,
// or accumulate adds to it
void launchAdjointPoints(const int inDims[3], const int outDims[3], int pad, const int32_t* adjMap, const int32_t* adjCell, int64_t V,
                         const float* contrib, float* out, int accumulate, hipStream_t s);
// processed-grid gradient -> input-grid gradient through padding / refinement
void launchPrepareAdjoint(const int inDims[3], const int outDims[3], int r, int pad, const float* dproc, float* din, int accumulate, hipStream_t s);

}  // namespace mdmc
