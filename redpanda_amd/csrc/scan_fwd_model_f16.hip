// The scan forward's instantiations (scan_fwd_kernel.h): the model's launches under fp16 autocast.
#include "scan_fwd_kernel.h"

namespace rp {
template hipError_t launch_scan_fwd_ty<kFwdModelF16>(int, int, int, const ScanParams&, const FwdOut&, hipStream_t);
}
