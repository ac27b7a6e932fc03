// The scan forward's launcher; the kernel is in scan_fwd_kernel.h, its
// instantiations in scan_fwd_*.hip (translation units of their own, compiled
// in parallel).

#include "redpanda_hip.h"
#include "rp_launch.h"

namespace rp {

// The instantiation for a launch's storage types: the combinations that the
// model and the scan's direct callers hand over have one each, any other mix
// shares kFwdAny.
hipError_t launch_scan_fwd(int S, int NPL, int gk, const ScanParams& p, const FwdOut& o,
                           hipStream_t st) {
  const int d = p.dt_delta, u = p.dt_u;
  const bool s_one = p.dt_B == p.dt_C;
  if (s_one && d == u && p.dt_B == u && !p.dsp && o.dcache == nullptr) {
    if (u == RP_F32) return launch_scan_fwd_ty<kFwdF32>(S, NPL, gk, p, o, st);
    if (u == RP_BF16) return launch_scan_fwd_ty<kFwdBf16>(S, NPL, gk, p, o, st);
    return launch_scan_fwd_ty<kFwdF16>(S, NPL, gk, p, o, st);
  }
  if (s_one && p.dt_B == RP_F32 && d == u && p.dsp) {
    if (u == RP_F32) return launch_scan_fwd_ty<kFwdF32Sp>(S, NPL, gk, p, o, st);
    if (u == RP_BF16) return launch_scan_fwd_ty<kFwdModelBf16>(S, NPL, gk, p, o, st);
    return launch_scan_fwd_ty<kFwdModelF16>(S, NPL, gk, p, o, st);
  }
  if (s_one && p.dt_B == RP_F32 && d == RP_F32 && u == RP_BF16 && !p.dsp && o.dcache == nullptr)
    return launch_scan_fwd_ty<kFwdMixBf16>(S, NPL, gk, p, o, st);
  return launch_scan_fwd_ty<kFwdAny>(S, NPL, gk, p, o, st);
}

}  // namespace rp
