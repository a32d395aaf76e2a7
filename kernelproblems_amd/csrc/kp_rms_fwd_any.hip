// Forward RMSNorm kernels for any width and alignment: instantiations.
#include "kp_rms_any.hpp"

namespace kp {
namespace rms {
namespace {

template <int LPR, int VPL, int WPR, int U>
FwdKernel for_terms(int nx) {
  switch (nx) {
    case 1: return rms_fwd_any<LPR, VPL, WPR, 1, U>;
    case 2: return rms_fwd_any<LPR, VPL, WPR, 2, U>;
    case 3: return rms_fwd_any<LPR, VPL, WPR, 3, U>;
  }
  return nullptr;
}

}  // namespace

FwdKernel fwd_any_kernel(const AnyShape& s, int nx) {
  switch (s.lpr * 100 + s.vpl * 10 + s.wpr) {
    case 811: return for_terms<8, 1, 1, 4>(nx);
    case 1611: return for_terms<16, 1, 1, 4>(nx);
    case 3211: return for_terms<32, 1, 1, 4>(nx);
    case 6411: return for_terms<64, 1, 1, 4>(nx);
    case 6421: return for_terms<64, 2, 1, 2>(nx);
    case 6422: return for_terms<64, 2, 2, 1>(nx);
    case 6424: return for_terms<64, 2, 4, 1>(nx);
    case 6434: return for_terms<64, 3, 4, 1>(nx);
    case 6444: return for_terms<64, 4, 4, 1>(nx);
    case 6454: return for_terms<64, 5, 4, 1>(nx);
    case 6464: return for_terms<64, 6, 4, 1>(nx);
    case 6474: return for_terms<64, 7, 4, 1>(nx);
    case 6484: return for_terms<64, 8, 4, 1>(nx);
  }
  return nullptr;
}

}  // namespace rms
}  // namespace kp
