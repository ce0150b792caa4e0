// forward_f64.hip -- FP64 instantiations of the forward kernels.
#include "forward_kernels.h"

namespace aw {

template int launch_fw<double, false>(const DevInst *, const FwTile *, int, void *, double *, size_t,
                                      hipStream_t, int, double, int *);
template int launch_fw<double, true>(const DevInst *, const FwTile *, int, void *, double *, size_t,
                                     hipStream_t, int, double, int *);

}  // namespace aw
