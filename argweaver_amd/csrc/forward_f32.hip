// forward_f32.hip -- FP32 instantiations of the forward kernels, and the
// check of FP32 tile starts.
#include "forward_kernels.h"

namespace aw {

template int launch_fw<float, false>(const DevInst *, const FwTile *, int, void *, double *, size_t,
                                     hipStream_t, int, double, int *);
template int launch_fw<float, true>(const DevInst *, const FwTile *, int, void *, double *, size_t,
                                    hipStream_t, int, double, int *);

int launch_fw_check(const DevInst *dD, const FwTile *tiles, const int *idx, int cnt,
                    const void *bnd, const double *bnorm, double tol, int *flags, hipStream_t st)
{
    hipLaunchKernelGGL(k_fw_check<float>, dim3(cnt), dim3(64), 0, st, dD, tiles, idx,
                       (const float *)bnd, bnorm, tol, flags);
    HIP_OK(hipGetLastError());
    return 0;
}

// LDS bytes of the forward kernel for R states per lane
size_t fw_lds_bytes(bool fp32, int R)
{
    auto one = [&](auto f32, auto f64) { return fp32 ? 4 * (size_t)f32 : 8 * (size_t)f64; };
    switch (R) {
    case 1: return one(fw_lds_reals<float, 1>(), fw_lds_reals<double, 1>());
    case 2: return one(fw_lds_reals<float, 2>(), fw_lds_reals<double, 2>());
    case 4: return one(fw_lds_reals<float, 4>(), fw_lds_reals<double, 4>());
    case 6: return one(fw_lds_reals<float, 6>(), fw_lds_reals<double, 6>());
    case 8: return one(fw_lds_reals<float, 8>(), fw_lds_reals<double, 8>());
    case 12: return one(fw_lds_reals<float, 12>(), fw_lds_reals<double, 12>());
    case 16: return one(fw_lds_reals<float, 16>(), fw_lds_reals<double, 16>());
    default: return one(fw_lds_reals<float, 32>(), fw_lds_reals<double, 32>());
    }
}

}  // namespace aw
