// Term combinations of rms_bwd_any: those of bwd_for_terms (without the fused
// forward + backward, which runs as two launches at these widths).
#pragma once

#include "kp_rms_any.hpp"

namespace kp {
namespace rms {

template <int LPR, int VPL, int WPR>
BwdKernel any_for_terms(int nx, int ndy, bool res) {
  if (!res) {
    if (nx == 1 && ndy == 1) return rms_bwd_any<LPR, VPL, WPR, 1, 1, false>;
    if (nx == 1 && ndy == 2) return rms_bwd_any<LPR, VPL, WPR, 1, 2, false>;
    if (nx == 1 && ndy == 3) return rms_bwd_any<LPR, VPL, WPR, 1, 3, false>;
    if (nx == 2 && ndy == 1) return rms_bwd_any<LPR, VPL, WPR, 2, 1, false>;
    if (nx == 3 && ndy == 1) return rms_bwd_any<LPR, VPL, WPR, 3, 1, false>;
    if (nx == 2 && ndy == 2) return rms_bwd_any<LPR, VPL, WPR, 2, 2, false>;
  } else {
    if (nx == 1 && ndy == 1) return rms_bwd_any<LPR, VPL, WPR, 1, 1, true>;
    if (nx == 1 && ndy == 2) return rms_bwd_any<LPR, VPL, WPR, 1, 2, true>;
    if (nx == 1 && ndy == 3) return rms_bwd_any<LPR, VPL, WPR, 1, 3, true>;
    if (nx == 2 && ndy == 2) return rms_bwd_any<LPR, VPL, WPR, 2, 2, true>;
  }
  return nullptr;
}

}  // namespace rms
}  // namespace kp
