// The scan backward's FAST instantiations: 4- and 8-lane shapes, the model's storage types.
#include "scan_bwd_fast_inst.h"

namespace rp {
template hipError_t launch_scan_bwd_fast<kBwdModel>(int, int, int, const ScanParams&, const BwdIO&, hipStream_t);
}
