// Definitions of the scan backward's FAST launchers (scan_bwd_kernel.h).  Each
// translation unit scan_bwd_fast*.hip instantiates one of them for one
// BwdTypes, so that they compile in parallel.
#pragma once

#include "scan_bwd_kernel.h"

namespace rp {

template <int TY>
hipError_t launch_scan_bwd_fast(int S, int NPL, int gk, const ScanParams& p, const BwdIO& io,
                                hipStream_t st) {
#define RP_CASE(SS, NN)                                                                \
  if (S == SS && NN == NPL)                                                            \
    return with_gate_kind_scan<SS, NN>(gk, [&](auto g) {                               \
      return launch_bwd_kernel<SS, NN, decltype(g), true, false, TY>(p, io, st);       \
    });
  RP_FOR_EACH_SHAPE_4_8(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

template <int TY>
hipError_t launch_scan_bwd_fast16(int S, int NPL, int gk, const ScanParams& p, const BwdIO& io,
                                  hipStream_t st) {
#define RP_CASE(SS, NN)                                                                \
  if (S == SS && NN == NPL)                                                            \
    return with_gate_kind_scan<SS, NN>(gk, [&](auto g) {                               \
      return launch_bwd_kernel<SS, NN, decltype(g), true, false, TY>(p, io, st);       \
    });
  RP_FOR_EACH_SHAPE_16(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

template <int TY>
hipError_t launch_scan_bwd_fast_walk(int S, int NPL, int gk, const ScanParams& p, const BwdIO& io,
                                     hipStream_t st) {
#define RP_CASE(SS, NN)                                                                \
  if (S == SS && NN == NPL)                                                            \
    return with_gate_kind_scan<SS, NN>(gk, [&](auto g) {                               \
      return launch_bwd_kernel<SS, NN, decltype(g), true, true, TY>(p, io, st);        \
    });
  RP_FOR_EACH_SHAPE_16(RP_CASE)
#undef RP_CASE
  return hipErrorInvalidValue;
}

}  // namespace rp
