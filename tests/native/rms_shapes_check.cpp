// Host check of the row shapes of kernelproblems_amd/csrc/kp_rms_shapes.hpp (the
// constexpr definitions the kernels compile): for every width the shapes take,
// each column is owned by exactly one lane element, every 16-byte chunk lies
// inside the row, and only the last chunk index is ever shifted or idle.
#include <cstdio>
#include <vector>

#include "kp_rms_shapes.hpp"

using namespace kp::rms;

static int check(int N, const AnyShape& s) {
  std::vector<int> owned(N, 0);
  int bad = 0;
  for (int part = 0; part < s.wpr; ++part)
    for (int sub = 0; sub < s.lpr; ++sub)
      for (int i = 0; i < s.vpl; ++i) {
        int start = any_col(i, part, sub, s.lpr, s.wpr), skip = 0;
        if (i == s.vpl - 1) {
          const AnyTail t = any_tail(start, N);
          start = t.start;
          skip = t.skip;
        }
        if (start < 0 || start + 8 > N || skip < 0 || skip > 8) ++bad;
        else
          for (int e = skip; e < 8; ++e) ++owned[start + e];
      }
  for (int c = 0; c < N; ++c) bad += owned[c] != 1;
  return bad;
}

int main() {
  int bad = 0;
  AnyShape s{};
  for (int64_t N = -1; N <= kAnyMaxN + 9; ++N) {
    const bool in = N >= kAnyMinN && N <= kAnyMaxN;
    for (int64_t M : {(int64_t)1, (int64_t)1 << 20}) {
      if (any_fwd_shape(M, N, 256, &s) != in) ++bad;
      else if (in && (check((int)N, s) != 0 || 4 % s.wpr != 0 || s.u < 1)) ++bad, std::printf("forward N=%d\n", (int)N);
    }
    if (any_loop_shape(N, &s) != (N > 1024 && N <= 5120)) ++bad;
    else if (N > 1024 && N <= 5120 && (check((int)N, s) != 0 || 4 % s.wpr != 0 || s.vpl > 5)) ++bad, std::printf("loop N=%d\n", (int)N);
    if (any_bwd_shape(N, &s) != in) ++bad;
    else if (in && (check((int)N, s) != 0 || kAnyWaves % s.wpr != 0)) ++bad, std::printf("backward N=%d\n", (int)N);
  }
  std::printf("%d bad widths\n", bad);
  return bad != 0;
}
