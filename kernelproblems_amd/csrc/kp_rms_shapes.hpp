// Row shapes of the RMSNorm kernels for any width (kp_rms_any.hpp): which lanes
// hold which columns.  constexpr and free of HIP, so that the kernels and the
// host-side unit test (g++) run this one definition.
#pragma once

#include <stdint.h>

namespace kp {
namespace rms {

constexpr int64_t kAnyMinN = 8, kAnyMaxN = 16384;
constexpr int kAnyWaves = 8;  // waves per block of the backward

// First column of chunk i of lane `sub` (of lpr) of the row's wave `part` (of wpr).
constexpr int any_col(int i, int part, int sub, int lpr, int wpr) { return ((i * wpr + part) * lpr + sub) * 8; }

// The last chunk, nominally at column c of a row of N >= 8: where it is read,
// and how many of its leading elements another lane owns.
struct AnyTail {
  int start, skip;
};
constexpr AnyTail any_tail(int c, int N) {
  const int s = c < N - 8 ? c : N - 8;
  return AnyTail{s, c < N ? c - s : 8};
}

// Row shapes: every chunk index below VPL - 1 lies wholly inside the row, i.e.
// (VPL - 1) * 8 * LPR * WPR <= N.  Forward (4-wave blocks): lanes per row, chunks per lane, waves
// per row, rows in flight per lane group; backward (8-wave blocks) without
// the last.
struct AnyShape {
  int lpr, vpl, wpr, u;
};
// false: no shape (N outside [kAnyMinN, kAnyMaxN]).
constexpr bool any_fwd_shape(int64_t N, AnyShape* s) {
  if (N < kAnyMinN || N > kAnyMaxN) return false;
  if (N <= 64) *s = {8, 1, 1, 4};
  else if (N <= 128) *s = {16, 1, 1, 4};
  else if (N <= 256) *s = {32, 1, 1, 4};
  else if (N <= 512) *s = {64, 1, 1, 4};
  else if (N <= 1024) *s = {64, 2, 1, 2};
  else if (N <= 2048) *s = {64, 2, 2, 1};
  else *s = {64, (int)((N + 2047) / 2048), 4, 1};
  return true;
}
constexpr bool any_bwd_shape(int64_t N, AnyShape* s) {
  if (N < kAnyMinN || N > kAnyMaxN) return false;
  if (N <= 64) *s = {8, 1, 1, 1};
  else if (N <= 128) *s = {16, 1, 1, 1};
  else if (N <= 256) *s = {32, 1, 1, 1};
  else if (N <= 512) *s = {64, 1, 1, 1};
  else if (N <= 1024) *s = {64, 2, 1, 1};
  else if (N <= 2048) *s = {64, 2, 2, 1};
  else if (N <= 4096) *s = {64, 2, 4, 1};
  else if (N <= 8192) *s = {64, 2, 8, 1};
  else if (N <= 12288) *s = {64, 3, 8, 1};
  else *s = {64, 4, 8, 1};
  return true;
}

}  // namespace rms
}  // namespace kp
