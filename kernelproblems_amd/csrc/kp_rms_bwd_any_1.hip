// Backward RMSNorm kernels for any width and alignment, rows of up to 1024 columns: instantiations.
#include "kp_rms_any_bwd.hpp"

namespace kp {
namespace rms {

BwdKernel bwd_any_kernel_short(const AnyShape& s, int nx, int ndy, bool res) {
  switch (s.lpr * 100 + s.vpl * 10 + s.wpr) {
    case 811: return any_for_terms<8, 1, 1>(nx, ndy, res);
    case 1611: return any_for_terms<16, 1, 1>(nx, ndy, res);
    case 3211: return any_for_terms<32, 1, 1>(nx, ndy, res);
    case 6411: return any_for_terms<64, 1, 1>(nx, ndy, res);
    case 6421: return any_for_terms<64, 2, 1>(nx, ndy, res);
  }
  return nullptr;
}

}  // namespace rms
}  // namespace kp
