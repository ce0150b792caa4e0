// forward.h -- the forward kernels' tiles and launches.
#pragma once

#include <hip/hip_runtime.h>

#include "engine.h"

namespace aw {

// A forward tile: columns [c0, c1) of an instance computed by one workgroup.
// mode 0 starts from the prior at column 0.  mode 1 starts at c0 from a
// uniform vector and stores nothing before cs (a warm-up: the filter
// forgets its start).  mode 2 starts at c0 from the column held in boundary
// slot bin (written by the tile before).  A tile with bout >= 0 also
// computes column c1 into boundary slot bout, for the check of the next
// tile's start.
struct FwTile {
    int inst;
    int c0, cs, c1;
    int mode;
    int bout, bin;
};
constexpr int BND_STRIDE = 64 * 32;   // Reals per boundary slot (the largest row)

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
