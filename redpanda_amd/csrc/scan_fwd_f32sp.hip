// The scan forward's instantiations (scan_fwd_kernel.h): fp32 inputs with softplus on load (the model in fp32).
#include "scan_fwd_kernel.h"

namespace rp {
template hipError_t launch_scan_fwd_ty<kFwdF32Sp>(int, int, int, const ScanParams&, const FwdOut&, hipStream_t);
}
