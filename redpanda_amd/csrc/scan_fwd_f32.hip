// The scan forward's instantiations (scan_fwd_kernel.h): fp32 inputs.
#include "scan_fwd_kernel.h"

namespace rp {
template hipError_t launch_scan_fwd_ty<kFwdF32>(int, int, int, const ScanParams&, const FwdOut&, hipStream_t);
}
