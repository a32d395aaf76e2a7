// RMSNorm row kernels for every width from 8 to 16384 and any 2-byte
// alignment: the widths, row addresses and strides that rms_fwd_vec /
// rms_bwd_vec (N = 512 * k, 16-byte rows) do not take.
//
// Layout: a row belongs to LPR lanes of each of WPR waves, and chunk i of a
// lane is the 8 columns from ((i * WPR + part) * LPR + lane % LPR) * 8, so
// only the last chunk index i = VPL - 1 can pass the row's end.  Rows of up to
// 256 columns take 8, 16 or 32 lanes (LPR), a wave holding 64 / LPR rows:
// one wave per row would leave 3/4 of its lanes idle at N = 128.
//
// Row end: the chunk that crosses it is read as the row's last 8 elements
// (in bounds: N >= 8) and the elements that the previous lane also holds are
// left out of the sums and of the weight gradient; both lanes then store the
// same bits there.  All loads of a row complete before its first store (the
// row's sum needs them), so outputs may alias inputs row by row.  Chunks
// wholly past the end re-read the same 8 elements and store nothing.
//
// Loads and stores are 16 bytes at 2-byte alignment: an odd N shifts every
// row, and the hardware splits the accesses that cross a line.
//
// Both directions are bound by memory traffic.  Measured on MI355X per call
// of the tensor-level entry points, against the scalar one-block-per-row
// kernels that these shapes took before (2-byte accesses, every row read
// twice, the weight-gradient partials updated in memory):
//   add + norm forward [3001, 2880]        35.9 -> 12.3 us (5.6 TB/s)
//   forward + backward [65536, 128]       275   -> 19.7 us (two row kernels and the finalize, 84 MB)
//   backward of [2048, 11001]             338   -> 44.9 us
#pragma once

#include "kp_rms_shapes.hpp"
#include "kp_rmsnorm_kernels.hpp"

namespace kp {
namespace rms {

// A lane's column chunks: where each starts, and how many leading elements of
// the last one belong to the previous lane (8: wholly past the row's end).
template <int LPR, int VPL, int WPR>
struct AnyCols {
  int start[VPL];
  int skip;
  __device__ __forceinline__ AnyCols(int part, int sub, int N) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) start[i] = any_col(i, part, sub, LPR, WPR);
    const AnyTail t = any_tail(start[VPL - 1], N);
    start[VPL - 1] = t.start;
    skip = t.skip;
  }
  // Whether chunk i holds columns of the row.
  __device__ __forceinline__ bool on(int i) const { return i < VPL - 1 || skip < 8; }
};

// Weight chunks: contiguous weights and whole-chunk segments by one load, any
// other segmentation element by element.
template <int LPR, int VPL, int WPR>
__device__ __forceinline__ void any_weight(u32x4 (&wv)[VPL], const uint16_t* w, int64_t seg_len, int64_t seg_stride,
                                           const AnyCols<LPR, VPL, WPR>& cols, int64_t N) {
  if (w == nullptr) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) wv[i] = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // bf16 1.0
  } else if (seg_len >= N) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) wv[i] = ld16u(w + cols.start[i]);
  } else if (((seg_len | N) & 7) == 0) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) wv[i] = ld16u(w + w_index(cols.start[i], seg_len, seg_stride));
  } else {
#pragma unroll
    for (int i = 0; i < VPL; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t lo = w[w_index(cols.start[i] + 2 * e, seg_len, seg_stride)];
        const uint32_t hi = w[w_index(cols.start[i] + 2 * e + 1, seg_len, seg_stride)];
        wv[i][e] = lo | (hi << 16);
      }
  }
}

// ------------------------------------------------------------------ forward
// One-shot grid of 4-wave blocks; U rows per lane group, all their loads in
// flight before the first sum (short rows would otherwise have one load per
// lane in flight).  The weight is requested after the rows: both are in
// flight together, and a block's few rows do not repay waiting for it first.
// GATHER: term 0's row is the one that the row's id names (see RmsFwdArgs; one
// wave-uniform id per wave), read with cacheable loads and summed in the same
// order, so that a gathered row and the same row given directly agree bit for
// bit.
template <int LPR, int VPL, int WPR, int NX, int U, bool GATHER = false>
__global__ __launch_bounds__(kThreads) void rms_fwd_any(RmsFwdArgs a) {
  static_assert(LPR == 64 || (WPR == 1 && VPL == 1), "");
  static_assert(!GATHER || (LPR == 64 && NX == 1 && U == 1), "");
  constexpr int RW = 64 / LPR;  // rows per wave
  __shared__ float red[U][4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % WPR, rloc = wave / WPR;
  const int sub = lane % LPR, rsub = lane / LPR;
  const int N = (int)a.N;
  const AnyCols<LPR, VPL, WPR> cols(part, sub, N);
  const int64_t row0 = ((int64_t)blockIdx.x * (4 / WPR) + rloc) * (U * RW) + rsub;

  u32x4 raw[U][NX][VPL];
  bool id_ok = true;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int64_t row = clamp_row(row0 + u * RW, a.M);
    if constexpr (GATHER) {
      const int64_t id = a.idx_bytes == 8 ? static_cast<const int64_t*>(a.idx)[row]
                                          : (int64_t) static_cast<const int32_t*>(a.idx)[row];
      id_ok = id >= 0 && id < a.idx_rows;
      row = id_ok ? id : 0;
    }
#pragma unroll
    for (int t = 0; t < NX; ++t) {
      const uint16_t* p = a.x[t] + row * a.xs[t];
#pragma unroll
      for (int i = 0; i < VPL; ++i) raw[u][t][i] = GATHER ? ld16u(p + cols.start[i]) : ld16u_stream(p + cols.start[i]);
    }
  }
  u32x4 wv[VPL];
  any_weight<LPR, VPL, WPR>(wv, a.w, a.w_seg_len, a.w_seg_stride, cols, a.N);
  __builtin_amdgcn_sched_barrier(0);

  u32x4 hv[U][VPL];
  float ss[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    ss[u] = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      u32x4 s = raw[u][0][i];
#pragma unroll
      for (int t = 1; t < NX; ++t) s = add_bf8(s, raw[u][t][i]);
      if (GATHER && !id_ok) s = u32x4{0u, 0u, 0u, 0u};
      hv[u][i] = s;
      float f[8];
      unpack8(s, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = (i < VPL - 1 || e >= cols.skip) ? f[e] : 0.f;
        ss[u] = fmaf(v, v, ss[u]);
      }
    }
    ss[u] = lanes_sum<LPR>(ss[u]);
  }
  if constexpr (WPR > 1) {
    if (lane == 0) {
#pragma unroll
      for (int u = 0; u < U; ++u) red[u][wave] = ss[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float t = 0.f;
#pragma unroll
      for (int p = 0; p < WPR; ++p) t += red[u][rloc * WPR + p];
      ss[u] = t;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t row = row0 + u * RW;
    if (row >= a.M) continue;
    const float r = 1.0f / sqrtf(ss[u] / (float)a.N + a.eps);
    uint16_t* yrow = a.y + row * a.ys;
    uint16_t* hrow = (NX > 1 || GATHER) && a.h != nullptr ? a.h + row * a.hs : nullptr;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float h[8], w[8], o[8];
      unpack8(hv[u][i], h);
      unpack8(wv[i], w);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (h[e] * r) * w[e];
      if (cols.on(i)) {
        st16u_stream(yrow + cols.start[i], pack8(o));
        if (hrow != nullptr) st16u_stream(hrow + cols.start[i], hv[u][i]);
      }
    }
    if (a.rstd != nullptr && part == 0 && sub == 0) a.rstd[row] = r;
    if (GATHER && !id_ok && part == 0 && sub == 0 && a.err) *a.err = 1;
  }
}

// The same for rows of middling width: persistent 4-wave blocks walking row
// groups grid-stride with the next group's loads in flight (two named register
// slots, unrolled two steps, as in rms_fwd_vec), the weight loaded once.
template <int VPL, int WPR, int NX>
__global__ __launch_bounds__(kThreads) void rms_fwd_any_loop(RmsFwdArgs a) {
  constexpr int RB = 4 / WPR;
  __shared__ float red[2][4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % WPR, rloc = wave / WPR;
  const AnyCols<64, VPL, WPR> cols(part, lane, (int)a.N);
  u32x4 wv[VPL];
  any_weight<64, VPL, WPR>(wv, a.w, a.w_seg_len, a.w_seg_stride, cols, a.N);
  int it = 0;
  auto load = [&](RawRow<VPL, NX>& s, int64_t row) {
    row = clamp_row(row, a.M);
#pragma unroll
    for (int t = 0; t < NX; ++t) {
      const uint16_t* p = a.x[t] + row * a.xs[t];
#pragma unroll
      for (int i = 0; i < VPL; ++i) s.v[t][i] = ld16u_stream(p + cols.start[i]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto proc = [&](const RawRow<VPL, NX>& s, int64_t row) {
    u32x4 hv[VPL];
    sum_raw<VPL, NX>(hv, s);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float f[8];
      unpack8(hv[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = (i < VPL - 1 || e >= cols.skip) ? f[e] : 0.f;
        ss = fmaf(v, v, ss);
      }
    }
    ss = wave_sum(ss);
    if constexpr (WPR > 1) {
      if (lane == 0) red[it & 1][wave] = ss;
      __syncthreads();
      float t = 0.f;
#pragma unroll
      for (int q = 0; q < WPR; ++q) t += red[it & 1][rloc * WPR + q];
      ss = t;
      ++it;
    }
    if (row >= a.M) return;
    const float r = 1.0f / sqrtf(ss / (float)a.N + a.eps);
    uint16_t* yrow = a.y + row * a.ys;
    uint16_t* hrow = NX > 1 && a.h != nullptr ? a.h + row * a.hs : nullptr;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float h[8], w[8], o[8];
      unpack8(hv[i], h);
      unpack8(wv[i], w);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = (h[e] * r) * w[e];
      if (cols.on(i)) {
        st16u_stream(yrow + cols.start[i], pack8(o));
        if (hrow != nullptr) st16u_stream(hrow + cols.start[i], hv[i]);
      }
    }
    if (a.rstd != nullptr && part == 0 && lane == 0) a.rstd[row] = r;
  };
  const int64_t G = gridDim.x, nb = block_trips(ceil_div_dev(a.M, RB), blockIdx.x, G);
  RawRow<VPL, NX> s0, s1;
  int64_t g = blockIdx.x, k = 0;
  load(s0, g * RB + rloc);
  for (; k + 2 < nb; k += 2, g += 2 * G) {
    load(s1, (g + G) * RB + rloc);
    proc(s0, g * RB + rloc);
    load(s0, (g + 2 * G) * RB + rloc);
    proc(s1, (g + G) * RB + rloc);
  }
  if (k + 1 < nb) {
    load(s1, (g + G) * RB + rloc);
    proc(s0, g * RB + rloc);
    proc(s1, (g + G) * RB + rloc);
  } else {
    proc(s0, g * RB + rloc);
  }
}

// ----------------------------------------------------------------- backward
// Persistent 8-wave blocks walking row groups grid-stride, the next group's
// loads in flight (two named register slots, unrolled two steps, as in
// rms_bwd_vec).  The column sums of the block's rows stay in registers; at
// the end its 8 / WPR x 64 / LPR row slots are added per column in slot order
// through LDS and written as one partial row, in rms_dw_finalize's layout.
// Rows of 12289 columns and more hold 4 chunks per lane: past 256 VGPRs with a
// second term or a residual, where the compiler spills 6 to 95 of them to
// scratch (a residual and three terms of 8193 to 12288 columns: 4).  They
// stay 6.6 to 11 times faster than the scalar kernel even so ([2048, 16384],
// one term 501 -> 50.6 us, two and two with a residual 1088 -> 128.5).
template <int VPL, int NX, int NDY, bool RES>
struct AnySlot {
  u32x4 x[NX][VPL], d[NDY][VPL], r[VPL];  // r: the residual gradient (RES)
  float q;
};

template <int LPR, int VPL, int WPR, int NX, int NDY, bool RES>
__device__ __forceinline__ void any_load(AnySlot<VPL, NX, NDY, RES>& s, const RmsBwdArgs& a, int64_t row,
                                         const AnyCols<LPR, VPL, WPR>& cols) {
  // the residual first: loads return in order, so a row's x and dy are not there before it (see any_row)
  if constexpr (RES)
#pragma unroll
    for (int i = 0; i < VPL; ++i) s.r[i] = ld16u_stream(a.dxr + row * a.dxrs + cols.start[i]);
#pragma unroll
  for (int t = 0; t < NX; ++t)
#pragma unroll
    for (int i = 0; i < VPL; ++i) s.x[t][i] = ld16u_stream(a.x[t] + row * a.xs[t] + cols.start[i]);
#pragma unroll
  for (int t = 0; t < NDY; ++t)
#pragma unroll
    for (int i = 0; i < VPL; ++i) s.d[t][i] = ld16u_stream(a.dy[t] + row * a.dys[t] + cols.start[i]);
  // without a given rstd the 4-byte load reads the row's first x word instead (never used): no load under a branch
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(a.x[0] + row * a.xs[0]) & ~(uintptr_t)3;
  s.q = *(a.rstd != nullptr ? a.rstd + row : reinterpret_cast<const float*>(x0));
}

template <int LPR, int VPL, int WPR, int NX, int NDY, bool RES>
__device__ __forceinline__ void any_row(const RmsBwdArgs& a, const AnySlot<VPL, NX, NDY, RES>& s,
                                        const u32x4 (&wv)[VPL], float (&acc)[VPL * 8],
                                        float (&red)[2][kAnyWaves][2], int64_t row,
                                        const AnyCols<LPR, VPL, WPR>& cols, int lane, int wave, int rloc, int it) {
  const bool have_rstd = a.rstd != nullptr;
  u32x4 xv[VPL], dv[VPL];
  float sxg = 0.f, ss = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    xv[i] = s.x[0][i];
#pragma unroll
    for (int t = 1; t < NX; ++t) xv[i] = add_bf8(xv[i], s.x[t][i]);
    dv[i] = s.d[0][i];
#pragma unroll
    for (int t = 1; t < NDY; ++t) dv[i] = add_bf8(dv[i], s.d[t][i]);
    float x[8], d[8], w[8];
    unpack8(xv[i], x);
    unpack8(dv[i], d);
    unpack8(wv[i], w);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      // elements of the previous lane are selected out, not multiplied out: they may be inf or NaN
      const bool own = i < VPL - 1 || e >= cols.skip;
      const float xe = own ? x[e] : 0.f, ge = own ? d[e] * w[e] : 0.f;
      sxg = fmaf(xe, ge, sxg);
      ss = fmaf(xe, xe, ss);
    }
  }
  // The residual has arrived before the row's barrier too: the lane before the
  // tail chunk may be another wave's, and dx may be written over the residual.
  u32x4 rv[VPL];
  if constexpr (RES) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      rv[i] = s.r[i];
      asm volatile("" : "+v"(rv[i]));
    }
  }
  sxg = lanes_sum<LPR>(sxg);
  if (!have_rstd) ss = lanes_sum<LPR>(ss);
  if constexpr (WPR > 1) {
    if (lane == 0) {
      red[it & 1][wave][0] = sxg;
      red[it & 1][wave][1] = ss;
    }
    __syncthreads();
    float t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int p = 0; p < WPR; ++p) {
      t0 += red[it & 1][rloc * WPR + p][0];
      t1 += red[it & 1][rloc * WPR + p][1];
    }
    sxg = t0;
    ss = t1;
  }
  const float r = have_rstd ? s.q : 1.0f / sqrtf(ss / (float)a.N + a.eps);
  const float cN = (r * sxg) * (1.0f / (float)a.N);
  if (row < a.M) {
    uint16_t* dxrow = a.dx + row * a.dxs;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float x[8], d[8], w[8], o[8];
      unpack8(xv[i], x);
      unpack8(dv[i], d);
      unpack8(wv[i], w);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float xh = x[e] * r;
        o[e] = (d[e] * w[e] - xh * cN) * r;
        acc[i * 8 + e] = fmaf(d[e], xh, acc[i * 8 + e]);  // a previous lane's element: never written out
      }
      u32x4 ov = pack8(o);
      if constexpr (RES) ov = add_bf8(rv[i], ov);
      if (cols.on(i)) st16u_stream(dxrow + cols.start[i], ov);
    }
  }
}

template <int LPR, int VPL, int WPR, int NX, int NDY, bool RES>
__global__ __launch_bounds__(kAnyWaves * 64) void rms_bwd_any(RmsBwdArgs a) {
  static_assert(LPR == 64 || (WPR == 1 && VPL == 1), "");
  constexpr int RW = 64 / LPR, RB = kAnyWaves / WPR, RS = RB * RW;  // rows per wave, per block of waves, per step
  constexpr int K = WPR * VPL * LPR * 8;                            // columns covered
  __shared__ float comb[RS > 1 ? RS * K : 1];
  __shared__ float red[2][kAnyWaves][2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % WPR, rloc = wave / WPR;
  const int sub = lane % LPR, slot = rloc * RW + lane / LPR;
  const int N = (int)a.N;
  const AnyCols<LPR, VPL, WPR> cols(part, sub, N);
  u32x4 wv[VPL];
  any_weight<LPR, VPL, WPR>(wv, a.w, a.w_seg_len, a.w_seg_stride, cols, a.N);
  float acc[VPL * 8];
#pragma unroll
  for (int j = 0; j < VPL * 8; ++j) acc[j] = 0.f;

  const int64_t G = gridDim.x, nb = block_trips(ceil_div_dev(a.M, RS), blockIdx.x, G);
  AnySlot<VPL, NX, NDY, RES> s0, s1;
  int it = 0;
  int64_t g = blockIdx.x, k = 0;
#define KP_LOAD(S, gg)                                                                  \
  any_load<LPR, VPL, WPR, NX, NDY, RES>(S, a, clamp_row((gg) * RS + slot, a.M), cols);  \
  __builtin_amdgcn_sched_barrier(0)
#define KP_PROC(S, gg)                                                                                              \
  any_row<LPR, VPL, WPR, NX, NDY, RES>(a, S, wv, acc, red, (gg) * RS + slot, cols, lane, wave, rloc, it);           \
  ++it
  KP_LOAD(s0, g);
  for (; k + 2 < nb; k += 2, g += 2 * G) {
    KP_LOAD(s1, g + G);
    KP_PROC(s0, g);
    KP_LOAD(s0, g + 2 * G);
    KP_PROC(s1, g + G);
  }
  if (k + 1 < nb) {
    KP_LOAD(s1, g + G);
    KP_PROC(s0, g);
    KP_PROC(s1, g + G);
  } else {
    KP_PROC(s0, g);
  }
#undef KP_LOAD
#undef KP_PROC
  if (a.partial == nullptr) return;
  if constexpr (RS == 1) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      if (!cols.on(i)) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (i < VPL - 1 || e >= cols.skip)
          a.partial[part_index(cols.start[i] + e, blockIdx.x, gridDim.x)] = acc[i * 8 + e];
    }
  } else {
    float* mine = comb + slot * K;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      if (!cols.on(i)) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (i < VPL - 1 || e >= cols.skip) mine[cols.start[i] + e] = acc[i * 8 + e];
    }
    __syncthreads();
    for (int c = threadIdx.x; c < N; c += kAnyWaves * 64) {
      float t = comb[c];
#pragma unroll
      for (int r = 1; r < RS; ++r) t += comb[r * K + c];
      a.partial[part_index(c, blockIdx.x, gridDim.x)] = t;
    }
  }
}

// Kernels for a shape and term counts, or nullptr (kp_rms_fwd_any.hip,
// kp_rms_bwd_any_1.hip, kp_rms_bwd_any_2.hip).
FwdKernel fwd_any_kernel(const AnyShape& s, int nx);
FwdKernel fwd_any_gather_kernel(const AnyShape& s);  // four waves per row, at most 8192 columns
FwdKernel fwd_any_loop_kernel(const AnyShape& s, int nx);
BwdKernel bwd_any_kernel_short(const AnyShape& s, int nx, int ndy, bool res);
BwdKernel bwd_any_kernel_wide(const AnyShape& s, int nx, int ndy, bool res);
inline BwdKernel bwd_any_kernel(const AnyShape& s, int nx, int ndy, bool res) {
  return s.wpr == 1 ? bwd_any_kernel_short(s, nx, ndy, res) : bwd_any_kernel_wide(s, nx, ndy, res);
}

}  // namespace rms
}  // namespace kp
