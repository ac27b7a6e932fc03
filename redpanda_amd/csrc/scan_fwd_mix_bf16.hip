// The scan forward's instantiations (scan_fwd_kernel.h): fp32 delta, B and C with bf16 u.
#include "scan_fwd_kernel.h"

namespace rp {
template hipError_t launch_scan_fwd_ty<kFwdMixBf16>(int, int, int, const ScanParams&, const FwdOut&, hipStream_t);
}
