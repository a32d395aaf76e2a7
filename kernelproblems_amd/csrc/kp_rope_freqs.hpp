// Inverse frequencies of rotary embedding from theta, evaluated on the host
// once per call.  Free of HIP, so that the host-side unit test (g++) runs this
// one definition.
#pragma once

#include <math.h>

namespace kp {

// inv[f] = fp32(theta^(-2f/D)), f < D / 2, as r^(f mod 16) q^(f / 16) with
// r = theta^(-2/D) and q = theta^(-32/D): two powers in place of D / 2.  The
// products are within about 40 fp64 roundings, 2^-47 relative, so an fp32
// value differs from the exactly rounded one only where that lies within
// 2^-23 of a unit of a tie.
inline void fill_inv_freq(double theta, int D, float* inv) {
  double lo[16] = {1.0, pow(theta, -2.0 / (double)D)};
  for (int i = 2; i < 16; ++i) lo[i] = lo[i / 2] * lo[i - i / 2];
  const double q = D > 32 ? pow(theta, -32.0 / (double)D) : 1.0;
  double hi = 1.0;
  for (int f = 0; f < D / 2; f += 16, hi *= q)
    for (int i = 0; i < 16 && f + i < D / 2; ++i) inv[f + i] = (float)(hi * lo[i]);
}

}  // namespace kp
