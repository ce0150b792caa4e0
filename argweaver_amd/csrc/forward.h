// forward.h -- the forward kernels' tiles and launches.
#pragma once

#include <hip/hip_runtime.h>

#include "engine.h"
#include "fw_plan.h"

namespace aw {

// LDS bytes of the forward kernel for R states per lane
size_t fw_lds_bytes(bool fp32, int R);

// Launch of cnt forward tiles on stream st.  BIG: the tiles of the instances
// with 32 states per lane.  early != null: re-run tiles (FP32 only), each
// reporting the column after the one that rejoined its stored columns, or 0.
template <class Real, bool BIG>
int launch_fw(const DevInst *dD, const FwTile *tiles, int cnt, void *bnd, double *bnorm, size_t sh,
              hipStream_t st, int T1max, double tol = 0.0, int *early = nullptr);

// launch of the checks of cnt speculative tile starts
int launch_fw_check(const DevInst *dD, const FwTile *tiles, const int *idx, int cnt,
                    const void *bnd, const double *bnorm, double tol, int *flags, hipStream_t st);

}  // namespace aw
