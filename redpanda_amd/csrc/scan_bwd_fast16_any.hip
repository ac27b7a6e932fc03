// The scan backward's FAST instantiations: 16-lane shapes, any storage types.
#include "scan_bwd_fast_inst.h"

namespace rp {
template hipError_t launch_scan_bwd_fast16<kBwdAny>(int, int, int, const ScanParams&, const BwdIO&, hipStream_t);
}
