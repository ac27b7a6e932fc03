// The general scan backward's tile-walking (MULTI) instantiations for the
// 16-lane shapes (kernel in scan_bwd_kernel.h): a workgroup walks io.tpw
// adjacent 16-channel tiles, whose dB / dC partials add into one block.  A
// translation unit of its own, compiled in parallel with the others.

#include "scan_bwd_kernel.h"

namespace rp {

hipError_t launch_scan_bwd_walk(int S, int NPL, int gk, const ScanParams& p, const BwdIO& io,
                                hipStream_t st) {
#define RP_CASE(SS, NN)                                                              \
  if (S == SS && NN == NPL)                                                          \
    return with_gate_kind_scan<SS, NN>(gk, [&](auto g) {                             \
      return launch_bwd_kernel<SS, NN, decltype(g), false, true, kBwdAny>(p, io, st); \
    });
  RP_FOR_EACH_SHAPE_16(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

}  // namespace rp
