// The pad-state instantiations of the step tile kernel (step_tile.h) for the
// 16-lane shapes: a translation unit of their own, compiled in parallel with
// the others in step_pad.hip.

#include "step_tile.h"

namespace rp {

hipError_t launch_step_tile_pad16(int S, int NPL, int gk, const StepParams& p, hipStream_t st) {
#define RP_CASE(SS, NN) \
  if (S == SS && NN == NPL) return launch_step_tile<SS, NN, true>(gk, p, st);
  RP_FOR_EACH_SHAPE_16(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

}  // namespace rp
