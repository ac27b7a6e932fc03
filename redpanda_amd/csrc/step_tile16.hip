// The step tile kernel's 16-lane shapes (step_tile.h): a translation unit of
// their own, compiled in parallel with the 4- and 8-lane ones in step.hip.

#include "step_tile.h"

namespace rp {

hipError_t launch_step_tile16(int S, int NPL, int gk, const StepParams& p, hipStream_t st) {
#define RP_CASE(SS, NN) \
  if (S == SS && NN == NPL) return launch_step_tile<SS, NN, false>(gk, p, st);
  RP_FOR_EACH_SHAPE_16(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

}  // namespace rp
