// Host check of kernelproblems_amd/csrc/kp_rope_freqs.hpp: every head width, the
// usual thetas and unusual ones, against long double powers rounded once.
#include <cmath>
#include <cstdio>
#include <initializer_list>

#include "kp_rope_freqs.hpp"

int main() {
  long checked = 0, differ = 0, bad = 0;
  float inv[256];
  for (double theta : {10000.0, 500000.0, 1000000.0, 10.0, 1.0, 0.5, 123456.789, 1e12})
    for (int D = 2; D <= 512; D += 2) {
      kp::fill_inv_freq(theta, D, inv);
      for (int f = 0; f < D / 2; ++f) {
        const long double exact = powl((long double)theta, -(long double)(2 * f) / (long double)D);
        const float want = (float)exact;
        const long double unit = ldexpl(1.0L, ilogbl(exact) - 23);
        ++checked;
        differ += inv[f] != want;
        if (fabsl((long double)inv[f] - exact) > unit * (0.5L + 0x1p-23L)) {
          ++bad;
          std::printf("theta %g D %d f %d: %.9g, exact %.12Lg\n", theta, D, f, inv[f], exact);
        }
      }
    }
  std::printf("%ld checked, %ld rounded the other way, %ld bad\n", checked, differ, bad);
  return bad != 0;
}
