// Inverse frequencies of rotary embedding from theta, evaluated on the host
// once per call.  Free of HIP, so that the host-side unit test (g++) runs this
// one definition.
#pragma once

#include <math.h>

namespace kp {

// inv[f] = fp32(theta^(-2f/D)), f < D / 2, as r^(f mod 16) theta^(-2 (f - f mod 16) / D)
// with r = theta^(-2/D): 1 + (D - 1) / 32 powers in place of D / 2.  The
// products are within about 25 fp64 roundings, 2^-48 relative, so an fp32
// value differs from the exactly rounded one only where that lies within
// 2^-24 of a unit of a tie.
inline void fill_inv_freq(double theta, int D, float* inv) {
  double lo[16] = {1.0, pow(theta, -2.0 / (double)D)};
  for (int i = 2; i < 16; ++i) lo[i] = lo[i / 2] * lo[i - i / 2];
  double hi = 1.0;
  for (int f = 0; f < D / 2; ++f) {
    if (f != 0 && (f & 15) == 0) hi = pow(theta, -(double)(2 * f) / (double)D);
    inv[f] = (float)(hi * lo[f & 15]);
  }
}

}  // namespace kp
