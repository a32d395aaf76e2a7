// Backward RMSNorm kernels for any width and alignment, rows split over several waves: instantiations.
#include "kp_rms_any_bwd.hpp"

namespace kp {
namespace rms {

BwdKernel bwd_any_kernel_wide(const AnyShape& s, int nx, int ndy, bool res) {
  switch (s.lpr * 100 + s.vpl * 10 + s.wpr) {
    case 6422: return any_for_terms<64, 2, 2>(nx, ndy, res);
    case 6424: return any_for_terms<64, 2, 4>(nx, ndy, res);
    case 6428: return any_for_terms<64, 2, 8>(nx, ndy, res);
    case 6438: return any_for_terms<64, 3, 8>(nx, ndy, res);
    case 6448: return any_for_terms<64, 4, 8>(nx, ndy, res);
  }
  return nullptr;
}

}  // namespace rms
}  // namespace kp
