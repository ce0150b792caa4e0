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

size_t fw_lds_bytes(bool fp32, int R)
{
    switch (R) {
    case 1: return fp32 ? sizeof(FwShared<float, 1>) : sizeof(FwShared<double, 1>);
    case 2: return fp32 ? sizeof(FwShared<float, 2>) : sizeof(FwShared<double, 2>);
    case 4: return fp32 ? sizeof(FwShared<float, 4>) : sizeof(FwShared<double, 4>);
    case 6: return fp32 ? sizeof(FwShared<float, 6>) : sizeof(FwShared<double, 6>);
    case 8: return fp32 ? sizeof(FwShared<float, 8>) : sizeof(FwShared<double, 8>);
    case 12: return fp32 ? sizeof(FwShared<float, 12>) : sizeof(FwShared<double, 12>);
    case 16: return fp32 ? sizeof(FwShared<float, 16>) : sizeof(FwShared<double, 16>);
    default: return fp32 ? sizeof(FwShared<float, 32>) : sizeof(FwShared<double, 32>);
    }
}

}  // namespace aw
