// The scan forward's instantiations (scan_fwd_kernel.h): any storage types.
#include "scan_fwd_kernel.h"

namespace rp {
template hipError_t launch_scan_fwd_ty<kFwdAny>(int, int, int, const ScanParams&, const FwdOut&, hipStream_t);
}
