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
// (VPL - 1) * 8 * LPR * WPR <= N.  Lanes per row, chunks per lane, waves per
// row and rows in flight per lane group (one-shot forward); 4-wave blocks
// forward, 8-wave blocks backward.
struct AnyShape {
  int lpr, vpl, wpr, u;
};
// One-shot forward of `rows` input rows (M times the terms).  false: no shape
// (N outside [kAnyMinN, kAnyMaxN]).  Short rows take several per lane group
// once that still leaves four blocks' input for each of cus CUs: [65536, 128]
// 6.9 us with four and 7.1 with one, [32768, 128] of two terms 6.4 and 7.7,
// but [16384, 128] 4.1 and 3.6, [2048, 500] 3.8 and 3.3.
constexpr bool any_fwd_shape(int64_t rows, int64_t N, int cus, AnyShape* s) {
  if (N < kAnyMinN || N > kAnyMaxN) return false;
  if (N <= 64) *s = {8, 1, 1, 4};
  else if (N <= 128) *s = {16, 1, 1, 4};
  else if (N <= 256) *s = {32, 1, 1, 4};
  else if (N <= 512) *s = {64, 1, 1, 4};
  else if (N <= 1024) *s = {64, 2, 1, 2};
  else if (N <= 2048) *s = {64, 2, 2, 1};
  else *s = {64, (int)((N + 2047) / 2048), 4, 1};
  if (rows < (int64_t)4 * cus * (4 / s->wpr) * (64 / s->lpr) * s->u) s->u = 1;
  return true;
}
// Persistent forward: one wave per row, or two, of at most 5 chunks per lane.
constexpr bool any_loop_shape(int64_t N, AnyShape* s) {
  if (N <= 1024 || N > 5120) return false;
  const int wpr = N <= 2560 ? 1 : 2;
  *s = {64, (int)((N + 512 * wpr - 1) / (512 * wpr)), wpr, 1};
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
