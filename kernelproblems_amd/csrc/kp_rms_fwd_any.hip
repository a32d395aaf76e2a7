// Forward RMSNorm kernels for any width and alignment: instantiations.
#include "kp_rms_any.hpp"

namespace kp {
namespace rms {
namespace {

template <int LPR, int VPL, int WPR, int U>
FwdKernel for_u(int nx) {
  switch (nx) {
    case 1: return rms_fwd_any<LPR, VPL, WPR, 1, U>;
    case 2: return rms_fwd_any<LPR, VPL, WPR, 2, U>;
    case 3: return rms_fwd_any<LPR, VPL, WPR, 3, U>;
  }
  return nullptr;
}
template <int LPR, int VPL, int WPR, int U>
FwdKernel for_terms(int u, int nx) {
  if constexpr (U > 1) {
    if (u > 1) return for_u<LPR, VPL, WPR, U>(nx);
  }
  return for_u<LPR, VPL, WPR, 1>(nx);
}
template <int VPL, int WPR>
FwdKernel loop_for(int nx) {
  switch (nx) {
    case 1: return rms_fwd_any_loop<VPL, WPR, 1>;
    case 2: return rms_fwd_any_loop<VPL, WPR, 2>;
    case 3: return rms_fwd_any_loop<VPL, WPR, 3>;
  }
  return nullptr;
}

}  // namespace

FwdKernel fwd_any_kernel(const AnyShape& s, int nx) {
  switch (s.lpr * 100 + s.vpl * 10 + s.wpr) {
    case 811: return for_terms<8, 1, 1, 4>(s.u, nx);
    case 1611: return for_terms<16, 1, 1, 4>(s.u, nx);
    case 3211: return for_terms<32, 1, 1, 4>(s.u, nx);
    case 6411: return for_terms<64, 1, 1, 4>(s.u, nx);
    case 6421: return for_terms<64, 2, 1, 2>(s.u, nx);
    case 6422: return for_terms<64, 2, 2, 1>(s.u, nx);
    case 6424: return for_terms<64, 2, 4, 1>(s.u, nx);
    case 6434: return for_terms<64, 3, 4, 1>(s.u, nx);
    case 6444: return for_terms<64, 4, 4, 1>(s.u, nx);
    case 6454: return for_terms<64, 5, 4, 1>(s.u, nx);
    case 6464: return for_terms<64, 6, 4, 1>(s.u, nx);
    case 6474: return for_terms<64, 7, 4, 1>(s.u, nx);
    case 6484: return for_terms<64, 8, 4, 1>(s.u, nx);
  }
  return nullptr;
}

FwdKernel fwd_any_gather_kernel(const AnyShape& s) {
  switch (s.lpr * 100 + s.vpl * 10 + s.wpr) {
    case 6424: return rms_fwd_any<64, 2, 4, 1, 1, true>;
    case 6434: return rms_fwd_any<64, 3, 4, 1, 1, true>;
    case 6444: return rms_fwd_any<64, 4, 4, 1, 1, true>;
  }
  return nullptr;
}

FwdKernel fwd_any_loop_kernel(const AnyShape& s, int nx) {
  switch (s.vpl * 10 + s.wpr) {
    case 31: return loop_for<3, 1>(nx);
    case 41: return loop_for<4, 1>(nx);
    case 51: return loop_for<5, 1>(nx);
    case 32: return loop_for<3, 2>(nx);
    case 42: return loop_for<4, 2>(nx);
    case 52: return loop_for<5, 2>(nx);
  }
  return nullptr;
}

}  // namespace rms
}  // namespace kp
