// Cross-entropy loss over a vocabulary for gfx950: the _log_softmax +
// nll_loss region at the end of a Llama step, forward and backward.
//
// Forward (sum reduction, ignore_index):
//   lse_i  = max_j x_ij + log(sum_j exp(x_ij - max_j x_ij))     x = fp32(bf16 logits)
//   loss   = scale * sum_{i: t_i != ignore} (lse_i - x_{i, t_i}),  total_weight = #{i: t_i != ignore}
// The log-softmax matrix itself is never materialised: each logits row is
// read once (HBM read-bound) with a running reference exponent and a sum of
// exponentials per lane, one wave per row.  Per-row losses land in a workspace and a
// second one-block launch sums them in a fixed order in fp64 (deterministic,
// no atomics).
//
// Backward, given the saved fp32 log-softmax L and the upstream gradient g of
// the summed loss:
//   out_ij = bf16( grad_ij - exp(L_ij) * s_i ),   grad_ij = (j == t_i) ? -g : 0,  s_i = sum_j grad_ij
// (nll_loss_backward then _log_softmax_backward_data, fp32, then _to_copy):
// a streaming kernel, 4 bytes read and 2 written per element, evaluated in
// the same fp32 operations as torch's kernels (expf, this order).
//
// Forward and backward straight from the bf16 logits (the whole region when
// the log-softmax is not needed elsewhere): one block per row holds the row
// in registers, so each logit is read once and each gradient written once.
#include <math.h>

#include "kp_common.hpp"
#include "kp_internal.hpp"

namespace kp {
namespace {

constexpr float kLog2e = 1.4426950408889634f;
constexpr int kThreads = 256;
constexpr int kWavesPerBlock = kThreads / kWave;

__device__ __forceinline__ int64_t target_at(const void* t, int bytes, int64_t i) {
  return bytes == 8 ? static_cast<const int64_t*>(t)[i] : (int64_t) static_cast<const int32_t*>(t)[i];
}

// ------------------------------------------------------------------ forward
struct FwdArgs {
  const uint16_t* logits;
  int64_t rs;  // row stride, elements
  int64_t M, V;
  const void* targets;
  int tbytes;
  int64_t ignore;
  double* row_loss;   // [M]: lse_i - x_{i,t_i}, 0 for ignored rows
  int32_t* row_valid;  // [M]: 1 when the row counts
  float* lse_out;     // optional [M]
  int32_t* err;       // optional flag: a target outside [0, V) and not ignore_index
};

// A lane's running state is (R, s): R an fp32 reference exponent in log2
// units (the running max times L, L = log2 e rounded to fp32, rounded to
// fp32) and s = sum_j 2^(x_j L - R), each exponent argument formed by one
// fma, so it is rounded once relative to its own size.  The row's
// log2(sum_j 2^(x_j L)) is R + log2(s), and lse = (R + log2 s) / L in fp64:
// dividing by the same L the exponents used makes the dominant term exact,
// so neither R's rounding (~2e-3 in log2 units at |max| ~ 3e4) nor L's
// (L = log2 e (1 - 1.3e-8)) scales with the logits' magnitude; what remains
// is ~1.3e-8 log(V) plus the fp32 sums.

// (R, s) folded with 8 more values.
__device__ __forceinline__ void online8(float& R, float& s, const float* v) {
  const float cm = fmaxf(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])), fmaxf(fmaxf(v[4], v[5]), fmaxf(v[6], v[7])));
  const float rn = fmaxf(R, cm * kLog2e);  // rounding to fp32 is monotone: max commutes with it
  if (rn == -INFINITY) {                   // nothing but -inf so far: (R, s) stays (-inf, 0), (-inf, NaN) if NaN among it
    const float t = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    if (t != t) s = t;
    return;
  }
  s *= (R == rn) ? 1.0f : __builtin_amdgcn_exp2f(R - rn);
  float c = 0.0f, d = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i += 2) {
    c += __builtin_amdgcn_exp2f(__builtin_fmaf(v[i], kLog2e, -rn));
    d += __builtin_amdgcn_exp2f(__builtin_fmaf(v[i + 1], kLog2e, -rn));
  }
  s += c + d;
  R = rn;
}

// (R1, s1) + (R2, s2) of two lanes' states; a NaN in s or R of either one is one in both lanes' sums.
__device__ __forceinline__ void combine(float& R, float& s, float R2, float s2) {
  const float rn = fmaxf(R, R2);
  if (rn == -INFINITY) {  // 0 + 0, or NaN
    R = rn;
    s += s2;
    return;
  }
  const float a = (R == rn) ? s : s * __builtin_amdgcn_exp2f(R - rn);
  const float b = (R2 == rn) ? s2 : s2 * __builtin_amdgcn_exp2f(R2 - rn);
  R = rn;
  s = a + b;
}

template <int CTRL>
__device__ __forceinline__ void combine_dpp(float& R, float& s) {
  combine(R, s, dpp_f<CTRL>(R), dpp_f<CTRL>(s));
}

// The row's target and the raw bf16 logit at it, requested by the row's wave
// before its data loads: the target is then a scalar load ahead of any store,
// and the logit's wait, at the end of the row, does not sit behind the row's
// stores (loaded after them, the two formed a chain of full waits on the
// kernel's last wave generation).  An id outside [0, V) reads column 0.
struct FwdTarget {
  int64_t t;
  uint16_t xt;
};
__device__ __forceinline__ FwdTarget row_target(const FwdArgs& a, int64_t row) {
  const int64_t t = target_at(a.targets, a.tbytes, row);
  const bool in = t >= 0 && t < a.V;
  return FwdTarget{t, a.logits[row * a.rs + (in ? t : 0)]};
}

// The states of the NT threads that share a row combined, identical in every
// one of them: lanes fold by DPP and readlane; the waves' states go through
// LDS (2 x NT / 64 floats), where the lanes of each wave fold them by DPP
// again, every 16-lane row the same (folding them one after another took each
// thread 15 steps of two exponentials a row at NT = 1024).
template <int NT>
__device__ __forceinline__ void row_combine(float& R, float& s, float* lds) {
  constexpr int W = NT / kWave;
  static_assert(W == 1 || W == 4 || W == 8 || W == 16, "");
  combine_dpp<0xB1>(R, s);   // quad_perm [1,0,3,2]
  combine_dpp<0x4E>(R, s);   // quad_perm [2,3,0,1]
  combine_dpp<0x141>(R, s);  // row_half_mirror
  combine_dpp<0x140>(R, s);  // row_mirror
  float r0 = readlane_f(R, 0), s0 = readlane_f(s, 0);
  combine(r0, s0, readlane_f(R, 16), readlane_f(s, 16));
  float r1 = readlane_f(R, 32), s1 = readlane_f(s, 32);
  combine(r1, s1, readlane_f(R, 48), readlane_f(s, 48));
  combine(r0, s0, r1, s1);
  R = r0;
  s = s0;
  if constexpr (W > 1) {
    const int w = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
    if (lane == 0) {
      lds[w] = R;
      lds[W + w] = s;
    }
    __syncthreads();
    R = lds[lane % W];
    s = lds[W + lane % W];
    combine_dpp<0xB1>(R, s);
    combine_dpp<0x4E>(R, s);
    if constexpr (W > 4) combine_dpp<0x141>(R, s);
    if constexpr (W > 8) combine_dpp<0x140>(R, s);
  }
}

// Row epilogue, by one lane: the row's loss from its combined state.
__device__ __forceinline__ void finish_row(const FwdArgs& a, int64_t row, FwdTarget rt, float R, float s) {
  const double lse = ((double)R + log2((double)s)) / (double)kLog2e;
  if (a.lse_out) a.lse_out[row] = (float)lse;
  const int64_t t = rt.t;
  int valid = t != a.ignore;
  if (valid && (t < 0 || t >= a.V)) {
    valid = 0;
    if (a.err) a.err[0] = 1;
  }
  a.row_loss[row] = valid ? lse - (double)bf_to_f(rt.xt) : 0.0;
  a.row_valid[row] = valid;
}

constexpr int kUnroll = 4;        // 16-byte chunks per lane per step (4 KiB per wave in flight)
constexpr float kStepMax = 0x1p64f;  // a step's sum of 2^(x log2 e - R) above this (or NaN) takes the exact path

// One step of a lane over kUnroll chunks.  Fast path: every exponential is
// taken against the lane's reference R as it stands, so there is no
// per-chunk max and no rescale; R only moves when a value exceeds it by more
// than 64 in log2 units (the step's sum passes 2^64), on the lane's first
// step (R = -inf makes every term +inf), or on inf / NaN input -- then the
// lane redoes the step exactly with online8, which moves R to the running
// max.  A stale (smaller) R only scales the lane's sum, which the (R, s)
// combines take into account.
//
// TAIL: the chunk that crosses the row's end is read as the row's last 8
// elements (V >= 8), and what the chunk before it holds of them, like every
// chunk past the end, counts as -inf.
template <int NT, bool TAIL>
__device__ __forceinline__ void fwd_step(const uint16_t* p, int64_t c0, int64_t V, int tid, float& R, float& s) {
  u32x4 v[kUnroll];
  int skip[kUnroll];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    const int64_t j = (c0 + u * NT + tid) * 8;
    const int64_t start = !TAIL || j < V - 8 ? j : V - 8;
    skip[u] = !TAIL ? 0 : j < V ? (int)(j - start) : 8;
    v[u] = ld16u_stream(p + start);
  }
  float f[kUnroll][8];
#pragma unroll
  for (int u = 0; u < kUnroll; ++u) {
    unpack8(v[u], f[u]);
    if (TAIL) {
#pragma unroll
      for (int i = 0; i < 8; ++i) f[u][i] = i < skip[u] ? -INFINITY : f[u][i];
    }
  }
  float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < kUnroll; ++u)
#pragma unroll
    for (int i = 0; i < 8; ++i) part[i & 3] += __builtin_amdgcn_exp2f(__builtin_fmaf(f[u][i], kLog2e, -R));
  const float step = (part[0] + part[1]) + (part[2] + part[3]);
  if (step <= kStepMax) {
    s += step;
  } else {
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) online8(R, s, f[u]);
  }
}

// NT threads per row (64: a wave, four rows a block; else a block per row),
// any stride and alignment, V >= 8: thread t reads chunks (k * NT + t) of 8
// elements, kUnroll per step, all loads of a step issued together.  Only the
// last step carries masks.
template <int NT>
__global__ __launch_bounds__(NT < kThreads ? kThreads : NT) void xent_fwd_vec(FwdArgs a) {
  __shared__ float red[2 * NT / kWave];
  const int64_t row = NT == kWave ? (int64_t)blockIdx.x * kWavesPerBlock +
                                        __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6))
                                  : (int64_t)blockIdx.x;
  if (row >= a.M) return;
  const FwdTarget rt = row_target(a, row);
  const int tid = NT == kWave ? threadIdx.x & (kWave - 1) : threadIdx.x;
  const uint16_t* p = a.logits + row * a.rs;
  constexpr int64_t kStep = (int64_t)kUnroll * NT;
  const int64_t full = a.V / 8 / kStep * kStep;
  float R = -INFINITY, s = 0.0f;
  for (int64_t c0 = 0; c0 < full; c0 += kStep) fwd_step<NT, false>(p, c0, a.V, tid, R, s);
  if (full * 8 < a.V) fwd_step<NT, true>(p, full, a.V, tid, R, s);
  row_combine<NT>(R, s, red);
  if (tid == 0) finish_row(a, row, rt, R, s);
}

// V < 8: lane l holds element l.
__global__ __launch_bounds__(kThreads) void xent_fwd_scalar(FwdArgs a) {
  const int64_t row = (int64_t)blockIdx.x * kWavesPerBlock + (threadIdx.x >> 6);
  if (row >= a.M) return;
  const FwdTarget rt = row_target(a, row);
  const int lane = threadIdx.x & (kWave - 1);
  float f[8] = {lane < a.V ? bf_to_f(a.logits[row * a.rs + lane]) : -INFINITY,
                -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY, -INFINITY};
  float R = -INFINITY, s = 0.0f;
  online8(R, s, f);
  row_combine<kWave>(R, s, nullptr);
  if (lane == 0) finish_row(a, row, rt, R, s);
}

// Sum of one double over the 64 lanes, the same tree and order as wave_sum.
template <int CTRL>
__device__ __forceinline__ double dpp_d(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, true);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double readlane_d(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ double row16_sum_d(double v) {
  v += dpp_d<0xB1>(v);
  v += dpp_d<0x4E>(v);
  v += dpp_d<0x141>(v);
  v += dpp_d<0x140>(v);
  return v;
}
__device__ __forceinline__ double wave_sum_d(double v) {
  v = row16_sum_d(v);
  return (readlane_d(v, 0) + readlane_d(v, 16)) + (readlane_d(v, 32) + readlane_d(v, 48));
}

// One block: loss = scale * sum(row_loss), total_weight = sum(row_valid), in a
// fixed order: thread t sums rows t, t + 1024, ... in fp64, four of them
// requested together (past the last row: the last one again, not added); lanes
// fold by DPP and readlane, then the 16 lanes of a DPP row fold the 16 wave
// sums (one barrier).  A chain of latencies, us at 64 / 2795 / 4096 / 16384 rows:
// 1.5 / 2.0 / 2.1 / 3.9; folding by __shfl_xor (an LDS round trip a step) and
// one load at a time below 4096 rows 2.5 / 3.2 / 3.8 / 4.8, a tree through LDS
// with a barrier per level 2.1 / 2.9 / 3.2 / 6.8.
constexpr int kFinThreads = 1024;
__global__ __launch_bounds__(kFinThreads) void xent_fwd_finish(const double* row_loss, const int32_t* row_valid,
                                                                int64_t M, double scale, float* loss, float* total_weight) {
  constexpr int kW = kFinThreads / kWave;
  static_assert(kW == 16, "");
  __shared__ double ls[kW], cs[kW];
  double acc = 0.0, cnt = 0.0;  // counts below 2^53 are exact in any order
  for (int64_t i = threadIdx.x; i < M; i += 4 * kFinThreads) {
    double l[4];
    int32_t c[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t r = i + k * kFinThreads < M ? i + k * kFinThreads : M - 1;
      l[k] = row_loss[r];
      c[k] = row_valid[r];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool in = i + k * kFinThreads < M;
      acc = in ? acc + l[k] : acc;
      cnt += in ? (double)c[k] : 0.0;
    }
  }
  acc = wave_sum_d(acc);
  cnt = wave_sum_d(cnt);
  const int lane = threadIdx.x & (kWave - 1);
  if (lane == 0) {
    ls[threadIdx.x >> 6] = acc;
    cs[threadIdx.x >> 6] = cnt;
  }
  __syncthreads();
  if (threadIdx.x >= kWave) return;
  acc = row16_sum_d(ls[lane & (kW - 1)]);
  cnt = row16_sum_d(cs[lane & (kW - 1)]);
  if (lane == 0) {
    loss[0] = (float)(acc * scale);
    total_weight[0] = (float)cnt;
  }
}

// ------------------------------------------------------------------ backward
struct BwdArgs {
  const float* lsm;
  int64_t rs;  // row stride of lsm, elements
  uint16_t* out;
  int64_t ors;  // row stride of out, elements
  int64_t M, V;
  const void* targets;
  int tbytes;
  int64_t ignore;
  float g;
  int32_t* err;
  int bpr;  // blocks per row (vector path)
};

// The row's target column and s_i = sum_j grad_ij (-g, or 0 for an ignored /
// out-of-range target).  Out-of-range targets raise the flag once per row.
__device__ __forceinline__ int64_t row_target(const BwdArgs& a, int64_t row, bool first, float& sum) {
  const int64_t t = target_at(a.targets, a.tbytes, row);
  const bool in_range = t >= 0 && t < a.V;
  if (t != a.ignore && !in_range && first && a.err) a.err[0] = 1;
  const bool valid = t != a.ignore && in_range;
  sum = valid ? -a.g : 0.0f;
  return valid ? t : -1;
}

// grad - expf(L) * s, as _log_softmax_backward_data evaluates it in fp32.
__device__ __forceinline__ float xent_grad(float l, bool is_target, float g, float sum) {
  const float grad = is_target ? -g : 0.0f;
  return grad - expf(l) * sum;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Rows of V = 4k elements, lsm rows 16-byte and out rows 8-byte aligned.  A
// block covers 2048 consecutive elements of one row (block b: row b / bpr,
// float4 groups [(b % bpr) * 512, +512)); wave w takes groups
// [w * 128, +128) as two 1 KiB load instructions (lane l: groups l and
// 64 + l) and writes each group's 4 bf16 as one 8-byte store.  Measured on
// MI355X for this 4-byte-read / 2-byte-write stream: one group per lane per
// instruction beats 2-4 (1086-1144 us at [8192, 128256] against 996 us), and
// lanes holding 8 consecutive elements (two loads 32 bytes apart, one
// 16-byte store) ran at 1144 us.
constexpr int64_t kBwdBlockGroups = (int64_t)kThreads * 2;  // float4 groups per block

__global__ __launch_bounds__(kThreads) void xent_bwd_vec(BwdArgs a) {
  const int64_t row = (int64_t)((int)blockIdx.x / a.bpr);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & (kWave - 1);
  const int64_t g0 = (int64_t)((int)blockIdx.x - (int)row * a.bpr) * kBwdBlockGroups + (int64_t)wave * 128;
  const int64_t gpr = a.V / 4;
  const f32x4* p = reinterpret_cast<const f32x4*>(a.lsm + row * a.rs);
  u32x2* q = reinterpret_cast<u32x2*>(a.out + row * a.ors);
  f32x4 v[2];
  int64_t gi[2];
  bool ok[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    gi[h] = g0 + h * kWave + lane;
    ok[h] = gi[h] < gpr;
    v[h] = __builtin_nontemporal_load(p + (ok[h] ? gi[h] : 0));
  }
  // The row's target after the data loads: its scalar load (lgkmcnt) is
  // waited for independently of the data (vmcnt), whereas ahead of them it
  // held every block's data loads back by a chain of scalar round trips.
  __builtin_amdgcn_sched_barrier(0);
  float sum;
  const int64_t t = row_target(a, row, g0 == 0 && lane == 0, sum);
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bool has = (t >> 2) == gi[h];  // t = -1 for rows without a target column
    float o[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = xent_grad(v[h][i], has && (t & 3) == i, a.g, sum);
    const u32x2 r = {pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3])};
    if (ok[h]) __builtin_nontemporal_store(r, q + gi[h]);
  }
}

__global__ __launch_bounds__(kThreads) void xent_bwd_scalar(BwdArgs a) {
  const int64_t total = a.M * a.V;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < total; i += (int64_t)gridDim.x * kThreads) {
    const int64_t r = i / a.V, j = i - r * a.V;
    float sum;
    const int64_t t = row_target(a, r, j == 0, sum);
    a.out[r * a.ors + j] = f_to_bf(xent_grad(a.lsm[r * a.rs + j], j == t, a.g, sum));
  }
}

// ------------------------------------------------------------------ forward + backward from the logits
// out_ij = bf16( grad_ij - exp(x_ij - lse_i) * s_i ) straight from the bf16
// logits (the _log_softmax -> nll_loss_forward -> nll_loss_backward ->
// _log_softmax_backward_data region with the fp32 log-softmax never stored),
// optionally with the forward's loss.  A row needs its lse before its first
// gradient, so a whole row is held on chip: NT threads per row, thread t
// holding chunks t + NT k (k < KC) in registers -- 16 chunks (64 VGPRs) of
// 1024 threads cover V <= 131072, e.g. the 128256-entry vocabulary (256 KB of
// bf16 per row).  Each element is read once and written once: 4 bytes per
// element instead of the 6 of a forward pass followed by a pass that re-reads
// the logits.  The lse comes from the same (R, s) states as the forward
// (exponents by one fma against R = fl(max L)), combined across the row's
// threads.
struct FbArgs {
  const uint16_t* logits;
  int64_t rs;  // row stride, elements
  uint16_t* out;
  int64_t ors;  // row stride of out, elements
  int64_t M, V;
  const void* targets;
  int tbytes;
  int64_t ignore;
  float g;             // upstream gradient of the summed loss
  double* row_loss;    // optional [M] (loss requested)
  int32_t* row_valid;  // optional [M]
  int32_t* err;
};

struct RowTarget {
  int64_t t;  // target column, -1 when the row has none
  bool valid;
};

__device__ __forceinline__ RowTarget fb_target_of(const FbArgs& a, int64_t t, int tid) {
  const bool in_range = t >= 0 && t < a.V;
  const bool valid = t != a.ignore && in_range;
  if (t != a.ignore && !in_range && tid == 0 && a.err) a.err[0] = 1;
  return RowTarget{valid ? t : -1, valid};
}

// One lane records the row's loss lse - x_t (x_t loaded before any store of
// the row, so out may alias the logits).  lse = (R + log2 s) / L with fp32
// log2 s (|log2 s| < 18 for V < 2^17: within 2^-24 x 18 of exact), summed and
// divided in fp64.
__device__ __forceinline__ void fb_row_loss(const FbArgs& a, int64_t row, const RowTarget& rt, float R, float s,
                                            float xt) {
  const double lse = ((double)R + (double)log2f(s)) / (double)kLog2e;
  a.row_loss[row] = rt.valid ? lse - (double)xt : 0.0;
  a.row_valid[row] = rt.valid;
}

// p g = exp(x - lse) g = 2^(x L - R) (g / s): the fma is rounded relative to
// x L - R (small for the large p), and k = g / s carries fp32 relative error.
// The target's entry is (p - 1) g with p = exp / s divided out first: p near 1
// (a confident row) has fp32 relative error, and p = 1 gives exactly 0.  A row
// without a target has k = 0 / s: 0, or NaN in every column where s is 0 or
// NaN (a row with NaN or +inf, or of -inf alone), as eager's 0 - p * 0.
__device__ __forceinline__ float fb_exp(float x, float R) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(x, kLog2e, -R));
}

__device__ __forceinline__ float fb_target_grad(float xt, float R, float s, float g) {
  return __builtin_fmaf(fb_exp(xt, R) / s, g, -g);
}

// Max of the bf16 values of KC packed chunks, as fp32.  bf16 values order as
// signed 16-bit integers while one of them is not negative: one packed max
// per two values instead of two unpacks and a max.  All negative: their order
// is that of unsigned integers reversed.
template <int KC>
__device__ __forceinline__ float packed_max(const u32x4* v) {
  typedef int16_t s16x2 __attribute__((ext_vector_type(2)));
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  s16x2 m = {INT16_MIN, INT16_MIN};
#pragma unroll
  for (int k = 0; k < KC; ++k)
#pragma unroll
    for (int d = 0; d < 4; ++d) m = __builtin_elementwise_max(m, __builtin_bit_cast(s16x2, (uint32_t)v[k][d]));
  const int16_t top = m[0] > m[1] ? m[0] : m[1];
  if (top >= 0) return bf_to_f((uint16_t)top);
  u16x2 n = {0xffff, 0xffff};
#pragma unroll
  for (int k = 0; k < KC; ++k)
#pragma unroll
    for (int d = 0; d < 4; ++d) n = __builtin_elementwise_min(n, __builtin_bit_cast(u16x2, (uint32_t)v[k][d]));
  return bf_to_f(n[0] < n[1] ? n[0] : n[1]);
}

// An empty asm that takes the packed chunks as in/out operands: the values
// unpacked in one pass cannot be reused in the next, so only the 4 x KC
// packed registers stay live across passes (reusing the 8 x KC unpacked
// floats needs twice the registers and spills at KC = 16).
template <int KC>
__device__ __forceinline__ void keep_packed(u32x4* v) {
#pragma unroll
  for (int k = 0; k < KC; ++k) asm volatile("" : "+v"(v[k]));
}

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// Word 3 0x00020000 is the raw-buffer setting of the gfx9 family (32-bit data
// format); loads past `bytes` return zeros.
__device__ __forceinline__ rsrc_t row_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// Target of `row` (int32 or int64 ids) by two 4-byte buffer loads and no
// branch: a load under a branch makes the wait-count pass drain every
// outstanding load and store at the join, i.e. the whole previous row's
// stores and this row's loads.  For int32 ids the high word may fall past
// the array, where the descriptor's range check returns 0.
__device__ __forceinline__ void fb_target_load(const FbArgs& a, int64_t row, uint32_t& lo, uint32_t& hi) {
  const rsrc_t r = row_rsrc(a.targets, (uint32_t)(a.M * a.tbytes));
  const uint32_t off = (uint32_t)(row * a.tbytes);
  lo = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0);
  hi = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off + 4u, 0, 0);
}
// The words pass through an empty asm first, so that the compiler neither
// sinks the high word's load into a branch nor reads the words before the
// row's own loads are issued.
__device__ __forceinline__ int64_t fb_target_value(const FbArgs& a, uint32_t lo, uint32_t hi) {
  asm volatile("" : "+v"(lo), "+v"(hi));
  return a.tbytes == 8 ? (int64_t)(((uint64_t)hi << 32) | lo) : (int64_t)(int32_t)lo;
}

// Chunks whose exponentials stay in fp32 registers from the sum to the
// gradient (8 registers in place of 4), as many as 128 VGPRs hold beside the
// packed ones; the others take theirs a second time.  Rows of several blocks
// a CU gain by it ([4096, 32000] 92.8 us with one kept, 90.0 us so); one row a
// CU waits for memory instead (NT = 1024, [8192, 128256]: 740 us with eight
// kept, 735 us with one).
constexpr int fb_kept(int nt, int kc) { return nt == 1024 ? 1 : kc < 12 ? kc : kc == 12 ? 11 : 24 - kc; }

// Any stride and alignment (16-byte accesses at 2-byte alignment from a
// scalar row base and a 32-bit offset), V >= 8, KC = ceil(ceil(V / 8) / NT):
// chunk k < KC - 1 of every thread lies inside the row.  The chunk that
// crosses the row's end is read as the row's last 8 elements; those that the
// chunk before it holds, like whole chunks past the end, are -inf for the max
// and the sum, and the rest are stored one by one.
//
// NT = 1024 (V > 65528) is persistent: one block per CU walks rows
// blockIdx.x, + gridDim.x, ...; the next row's loads are issued as soon as
// the previous row's stores are, so the store stream of one row overlaps the
// load stream of the next (754 us against 791 us for one fresh block per row
// at [8192, 128256]).  Issuing the next row's chunk k right after row r's
// chunk k is unpacked, interleaved with row r's stores, measured slower
// (808 us).  Shorter rows take fewer threads, so that several rows are in
// different phases on a CU.  The LDS slots of the row reduction alternate
// between rows (a slow wave may still read row r's slots while a fast one
// writes row r + 1's).
//
// Bound by HBM: a third less VALU work per element (packed maxima, the target
// and 1 / s out of the gradient's inner loop) only took [8192, 128256] from
// 752 to 735 us, of 640 us for a plain copy of its bytes -- a row's loads,
// reduction and stores follow one another on its CU.  Rows that are not
// 16-byte aligned cost 1.17x ([2048, 50257] 95.5 us, [2048, 50256] 81.7 us;
// the scalar two-pass kernel they took before 252 us); plain (write-back)
// stores or loads are slower at either alignment (97.9 and 97.3 us, and
// 85.4 and 82.5 us).  Threads by the row's length, against one persistent
// 1024-thread block per CU for every V: [4096, 32000] 123 -> 90 us,
// [8192, 8192] 142 -> 48 us, [8192, 1003] 28 us (scalar) -> 12.5 us.
template <int NT, int KC>
__global__ __launch_bounds__(NT < kThreads ? kThreads : NT, KC > 8 ? 4 : 1) void xent_fwd_bwd_vec(FbArgs a) {
  constexpr int kRows = NT < kThreads ? kThreads / NT : 1;
  constexpr int KE = fb_kept(NT, KC);
  __shared__ float red[2][2 * NT / kWave];
  const int V = (int)a.V, cpr = (V + 7) / 8;
  u32x4 v[KC];
  int parity = 0;
  const int64_t r0 = (int64_t)blockIdx.x * kRows +
                     (kRows > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0);
  for (int64_t row = r0; row < a.M; row += (int64_t)gridDim.x * kRows, parity ^= 1) {
    // the thread index passes through an empty asm each row, so the chunk
    // offsets derived from it are recomputed where they are used instead of
    // being hoisted out of the loop (16 more live VGPRs)
    int tid = kRows > 1 ? threadIdx.x & (kWave - 1) : threadIdx.x;
    asm volatile("" : "+v"(tid));
    // the row's target is requested ahead of its data: vmcnt counts in issue
    // order, so waiting for the target afterwards does not wait for the row
    uint32_t t_lo, t_hi;
    fb_target_load(a, row, t_lo, t_hi);
    __builtin_amdgcn_sched_barrier(0);
    const char* xr = reinterpret_cast<const char*>(a.logits + row * a.rs);
    int cl = tid + (KC - 1) * NT;  // the last chunk, where it starts and how much of it is another's
    int start = cl * 8 < V - 8 ? cl * 8 : V - 8;
    int skip = cl < cpr ? cl * 8 - start : 8;
#pragma unroll
    for (int k = 0; k < KC; ++k)
      v[k] = ld16u_stream(reinterpret_cast<const uint16_t*>(
          xr + (k < KC - 1 ? (uint32_t)(tid + k * NT) * 16u : (uint32_t)start * 2u)));
    __builtin_amdgcn_sched_barrier(0);
    const RowTarget rt = fb_target_of(a, fb_target_value(a, t_lo, t_hi), tid);
    // x_t, loaded by every lane without a branch (element 0 where there is no
    // target) and consumed only before the row reduction, so its wait is not
    // a wait for the whole row
    uint16_t xtb = *reinterpret_cast<const uint16_t*>(xr + (uint32_t)(rt.valid ? (int)rt.t : 0) * 2u);
    if (skip > 0) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const uint32_t m = (2 * d < skip ? 0xffffu : 0u) | (2 * d + 1 < skip ? 0xffff0000u : 0u);
        v[KC - 1][d] = (v[KC - 1][d] & ~m) | (0xff80ff80u & m);
      }
    }
    float R = packed_max<KC>(v) * kLog2e, s = 0.0f;
    keep_packed<KC>(v);
    float e[KE][8];
    const float Rl = R;
    {
      const float ref = R == -INFINITY ? 0.0f : R;  // nothing but -inf: every exponential is 0
      float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int k = 0; k < KC; ++k) {
        float f[8];
        unpack8(v[k], f);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const float x = fb_exp(f[i], ref);
          if (k < KE) e[k][i] = x;
          part[i & 3] += x;
        }
      }
      s = (part[0] + part[1]) + (part[2] + part[3]);
    }
    asm volatile("" : "+v"(xtb));  // x_t has arrived before the barrier: other waves may overwrite it after
    const float xt = bf_to_f(xtb);
    row_combine<NT>(R, s, red[parity]);
    if (a.row_loss != nullptr && tid == 0) fb_row_loss(a, row, rt, R, s, xt);
    const float kf = (rt.valid ? a.g : 0.0f) / s;
    const float kl = Rl == R ? kf : kf * __builtin_amdgcn_exp2f(Rl - R);  // for the kept exponentials, against Rl
    keep_packed<KC - KE>(v + KE);
    asm volatile("" : "+v"(tid));  // the store offsets are recomputed here, not kept from the loads
    char* out = reinterpret_cast<char*>(a.out + row * a.ors);
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      float o[8];
      if (k < KE) {
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = e[k][i] * kl;
      } else {
        float f[8];
        unpack8(v[k], f);
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = fb_exp(f[i], R) * kf;
      }
      if (k < KC - 1) {
        st16u_stream(reinterpret_cast<uint16_t*>(out + (uint32_t)(tid + k * NT) * 16u), pack8(o));
      } else {
        cl = tid + (KC - 1) * NT;
        start = cl * 8 < V - 8 ? cl * 8 : V - 8;
        skip = cl < cpr ? cl * 8 - start : 8;
        uint16_t* q = reinterpret_cast<uint16_t*>(out + (uint32_t)start * 2u);
        if (skip == 0) {
          st16u_stream(q, pack8(o));
        } else {
#pragma unroll
          for (int i = 1; i < 8; ++i)
            if (i >= skip) q[i] = f_to_bf(o[i]);
        }
      }
    }
    // the target's entry once more, by the thread that stored it above
    if (rt.valid && tid == ((int)rt.t >> 3) % NT)
      *reinterpret_cast<uint16_t*>(out + (uint32_t)rt.t * 2u) = f_to_bf(fb_target_grad(xt, R, s, a.g));
  }
}

// Rows wider than the register kernel holds (or V < 8): 256 threads per row,
// two passes over the row (the second re-reads it); each element is read
// before it is written by the same thread, so out may alias the logits here
// too.
__global__ __launch_bounds__(kThreads) void xent_fwd_bwd_scalar(FbArgs a) {
  __shared__ float red[2 * kWavesPerBlock];
  const int64_t row = blockIdx.x;
  const uint16_t* x = a.logits + row * a.rs;
  uint16_t* o = a.out + row * a.ors;
  const RowTarget rt = fb_target_of(a, target_at(a.targets, a.tbytes, row), threadIdx.x);
  const float xt = (a.row_loss != nullptr && threadIdx.x == 0 && rt.valid) ? bf_to_f(x[rt.t]) : 0.0f;
  float R = -INFINITY, s = 0.0f;
  for (int64_t j0 = 0; j0 < a.V; j0 += 8 * kThreads) {
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t j = j0 + i * kThreads + threadIdx.x;
      f[i] = j < a.V ? bf_to_f(x[j]) : -INFINITY;
    }
    online8(R, s, f);
  }
  asm volatile("" ::"v"(xt));  // x_t has arrived before the barrier: other waves may overwrite it after
  row_combine<kThreads>(R, s, red);
  if (a.row_loss != nullptr && threadIdx.x == 0) fb_row_loss(a, row, rt, R, s, xt);
  const float kf = (rt.valid ? a.g : 0.0f) / s;
  for (int64_t j = threadIdx.x; j < a.V; j += kThreads) {
    const float xj = bf_to_f(x[j]);
    o[j] = f_to_bf(j == rt.t ? fb_target_grad(xj, R, s, a.g) : fb_exp(xj, R) * kf);
  }
}

// The register kernel for rows of V elements: NT threads per row and KC
// chunks per thread, or false.
typedef void (*FbKernel)(FbArgs);
template <int NT, int KC, int KMAX>
FbKernel fb_pick(int kc) {
  if constexpr (KC > KMAX) return nullptr;
  else return kc == KC ? xent_fwd_bwd_vec<NT, KC> : fb_pick<NT, KC + 1, KMAX>(kc);
}
struct FbPlan {
  FbKernel kernel;
  int threads, rows;  // per block
  bool persistent;
};
FbPlan fb_plan(int64_t V) {
  const int64_t cpr = ceil_div(V, 8);
  if (V < 8 || cpr > 16 * 1024) return FbPlan{nullptr, 0, 0, false};
  if (cpr <= 512) return FbPlan{fb_pick<64, 1, 8>((int)ceil_div(cpr, 64)), kThreads, kThreads / 64, false};
  if (cpr <= 2048) return FbPlan{fb_pick<256, 3, 8>((int)ceil_div(cpr, 256)), 256, 1, false};
  if (cpr <= 8192) return FbPlan{fb_pick<512, 5, 16>((int)ceil_div(cpr, 512)), 512, 1, false};
  return FbPlan{fb_pick<1024, 9, 16>((int)ceil_div(cpr, 1024)), 1024, 1, true};
}

bool valid_target_bytes(int b) { return b == 4 || b == 8; }

// Threads per row of the forward: a wave while there are rows enough to fill
// the chip, else a block (a wave streams a row at a few GB/s by itself).  A
// block's start and reduction weigh the more the shorter the row, a second
// step of 256 threads (16384 elements each) that is less than half full idles,
// and rows at any address leave fewer lines in flight, so the line lies at 2,
// 3, 4 or 6 rows per CU.  Measured on MI355X (256 CUs), per call of both
// launches, a wave / 256 threads (us): V = 12288 512 rows 12.0 / 10.7, 768
// 12.2 / 12.3; 16384 1280 rows 16.2 / 15.3, 1600 16.6 / 17.4; 18432 768 rows
// 14.6 / 13.6, 1024 15.2 / 15.8, 1815 18.1 / 22.1; 24576 1536 20.4 / 18.5; 32768
// 1536 rows 25.8 / 22.2; 50256 1536 rows 34.4 / 33.4, 1600 34.7 / 36.9; 90880
// 1815 rows 57.3 / 63.2; rows not 16-byte aligned: 24577 1024 rows 19.5 /
// 18.6, 1152 21.5 / 21.9; 50257 1024 rows 31.8 / 28.7, 1408 35.3 / 38.4;
// 1024 threads, 256 / 1024: 128256 256 rows 26.6 / 18.1, 512 30.8 / 28.0, 768
// 37.9 / 37.7; 90880 512 rows 24.9 / 23.0; 18432 256 rows 10.5 / 11.2.
int fwd_threads(int64_t M, int64_t V, bool aligned, int cus) {
  const int64_t per_cu = V < 16384 ? 2 : V > 16384 && V < 24576 ? 3 : aligned ? 6 : 4;
  if (V < 8192 || M > per_cu * cus) return 64;
  return M < (int64_t)2 * cus && V >= 32768 ? 1024 : 256;
}

}  // namespace
}  // namespace kp

using namespace kp;

extern "C" {

size_t kp_cross_entropy_fwd_workspace_size(int64_t M) {
  if (M <= 0) return 0;
  return (size_t)M * sizeof(double) + (size_t)M * sizeof(int32_t);
}

int kp_cross_entropy_fwd_bf16(const void* logits, int64_t row_stride, int64_t M, int64_t V, const void* targets,
                              int target_bytes, int64_t ignore_index, float scale, float* loss, float* total_weight,
                              float* row_lse, int32_t* error_flag, void* workspace, size_t workspace_bytes,
                              void* stream) {
  static const char* who = "kp_cross_entropy_fwd_bf16";
  if (M < 0 || V < 1) return fail(KP_EINVAL, "%s: bad shape [%lld, %lld]", who, (long long)M, (long long)V);
  if (loss == nullptr || total_weight == nullptr) return fail(KP_EINVAL, "%s: loss / total_weight is NULL", who);
  if (!valid_target_bytes(target_bytes)) return fail(KP_EINVAL, "%s: target_bytes must be 4 or 8", who);
  if (M > 1 && row_stride < V) return fail(KP_EINVAL, "%s: row stride %lld < V", who, (long long)row_stride);
  const size_t need = kp_cross_entropy_fwd_workspace_size(M);
  if (M > 0 && (logits == nullptr || targets == nullptr)) return fail(KP_EINVAL, "%s: logits / targets NULL", who);
  if (workspace_bytes < need || (need && workspace == nullptr))
    return fail(KP_EWORKSPACE, "%s: workspace of %zu bytes needed", who, need);
  if ((reinterpret_cast<uintptr_t>(workspace) & 7) != 0) return fail(KP_EINVAL, "%s: workspace not 8-byte aligned", who);
  if (M > ((int64_t)1 << 31) * kWavesPerBlock) return fail(KP_EUNSUPPORTED, "%s: too many rows", who);
  hipStream_t st = as_stream(stream);
  FwdArgs a{};
  a.logits = static_cast<const uint16_t*>(logits);
  a.rs = row_stride;
  a.M = M;
  a.V = V;
  a.targets = targets;
  a.tbytes = target_bytes;
  a.ignore = ignore_index;
  a.row_loss = static_cast<double*>(workspace);
  a.row_valid = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + (size_t)M * sizeof(double));
  a.lse_out = row_lse;
  a.err = error_flag;
  if (M > 0) {
    const bool aligned = aligned16(logits) && (M == 1 || row_stride % 8 == 0);
    const int nt = V < 8 ? 0 : fwd_threads(M, V, aligned, cu_count());
    const void* fk = nt == 0     ? reinterpret_cast<const void*>(xent_fwd_scalar)
                     : nt == 64  ? reinterpret_cast<const void*>(xent_fwd_vec<64>)
                     : nt == 256 ? reinterpret_cast<const void*>(xent_fwd_vec<256>)
                                 : reinterpret_cast<const void*>(xent_fwd_vec<1024>);
    // Rows in slabs of what one launch takes (several only at a wave per row).
    constexpr int64_t kSlab = max_blocks(kThreads) * kWavesPerBlock;
    for (int64_t r0 = 0; r0 < M; r0 += kSlab) {
      FwdArgs b = a;
      b.M = M - r0 < kSlab ? M - r0 : kSlab;
      b.logits += r0 * row_stride;
      b.targets = static_cast<const char*>(targets) + r0 * target_bytes;
      b.row_loss += r0;
      b.row_valid += r0;
      if (row_lse != nullptr) b.lse_out += r0;
      const unsigned blocks = (unsigned)(nt > 64 ? b.M : ceil_div(b.M, kWavesPerBlock));
      void* args[] = {&b};
      launch_dominant_raw(fk, dim3(blocks), dim3(nt > kThreads ? nt : kThreads), args, 0, st);
      const int rc = check_launch(who);
      if (rc != KP_OK) return rc;
    }
  }
  hipLaunchKernelGGL(xent_fwd_finish, dim3(1), dim3(kFinThreads), 0, st, a.row_loss, a.row_valid, M, (double)scale,
                     loss, total_weight);
  return check_launch(who);
}

int kp_cross_entropy_bwd_bf16(const float* log_softmax, int64_t lsm_row_stride, const void* targets, int target_bytes,
                              int64_t ignore_index, float grad_loss, void* grad_logits, int64_t out_row_stride,
                              int64_t M, int64_t V, int32_t* error_flag, void* stream) {
  static const char* who = "kp_cross_entropy_bwd_bf16";
  if (M < 0 || V < 1) return fail(KP_EINVAL, "%s: bad shape [%lld, %lld]", who, (long long)M, (long long)V);
  if (!valid_target_bytes(target_bytes)) return fail(KP_EINVAL, "%s: target_bytes must be 4 or 8", who);
  if (M == 0) return KP_OK;
  if (log_softmax == nullptr || targets == nullptr || grad_logits == nullptr)
    return fail(KP_EINVAL, "%s: NULL operand", who);
  if (M > 1 && (lsm_row_stride < V || out_row_stride < V)) return fail(KP_EINVAL, "%s: row stride < V", who);
  if (M > (((int64_t)1 << 62) / V)) return fail(KP_EUNSUPPORTED, "%s: too large", who);
  BwdArgs a{};
  a.lsm = log_softmax;
  a.rs = lsm_row_stride;
  a.out = static_cast<uint16_t*>(grad_logits);
  a.ors = out_row_stride;
  a.M = M;
  a.V = V;
  a.targets = targets;
  a.tbytes = target_bytes;
  a.ignore = ignore_index;
  a.g = grad_loss;
  a.err = error_flag;
  const bool vec = V % 4 == 0 && aligned16(log_softmax) && (reinterpret_cast<uintptr_t>(grad_logits) & 7) == 0 &&
                   (M == 1 || (lsm_row_stride % 4 == 0 && out_row_stride % 4 == 0));
  void* args[] = {&a};
  const int64_t bpr = ceil_div(V, 4 * kBwdBlockGroups);  // blocks per row
  if (vec && bpr <= max_blocks(kThreads) / M) {
    a.bpr = (int)bpr;
    launch_dominant_raw(reinterpret_cast<const void*>(xent_bwd_vec), dim3((unsigned)(bpr * M)), dim3(kThreads), args,
                        0, as_stream(stream));
  } else {
    const int64_t want = ceil_div(M * V, kThreads);
    const int64_t cap = (int64_t)cu_count() * 16;
    launch_dominant_raw(reinterpret_cast<const void*>(xent_bwd_scalar), dim3((unsigned)(want < cap ? want : cap)),
                        dim3(kThreads), args, 0, as_stream(stream));
  }
  return check_launch(who);
}

int kp_cross_entropy_fwd_bwd_bf16(const void* logits, int64_t row_stride, int64_t M, int64_t V, const void* targets,
                                  int target_bytes, int64_t ignore_index, float grad_loss, void* grad_logits,
                                  int64_t out_row_stride, float scale, float* loss, float* total_weight,
                                  int32_t* error_flag, void* workspace, size_t workspace_bytes, void* stream) {
  static const char* who = "kp_cross_entropy_fwd_bwd_bf16";
  if (M < 0 || V < 1) return fail(KP_EINVAL, "%s: bad shape [%lld, %lld]", who, (long long)M, (long long)V);
  if (!valid_target_bytes(target_bytes)) return fail(KP_EINVAL, "%s: target_bytes must be 4 or 8", who);
  if ((loss == nullptr) != (total_weight == nullptr))
    return fail(KP_EINVAL, "%s: loss and total_weight are both given or both NULL", who);
  const bool want_loss = loss != nullptr;
  const size_t need = want_loss ? kp_cross_entropy_fwd_workspace_size(M) : 0;
  if (workspace_bytes < need || (need && workspace == nullptr))
    return fail(KP_EWORKSPACE, "%s: workspace of %zu bytes needed", who, need);
  if (need && (reinterpret_cast<uintptr_t>(workspace) & 7) != 0)
    return fail(KP_EINVAL, "%s: workspace not 8-byte aligned", who);
  if (M > 0 && (logits == nullptr || targets == nullptr || grad_logits == nullptr))
    return fail(KP_EINVAL, "%s: NULL operand", who);
  if (M > 1 && (row_stride < V || out_row_stride < V)) return fail(KP_EINVAL, "%s: row stride < V", who);
  if (M > 0x7fffffffLL) return fail(KP_EUNSUPPORTED, "%s: too many rows", who);
  hipStream_t st = as_stream(stream);
  FbArgs a{};
  a.logits = static_cast<const uint16_t*>(logits);
  a.rs = row_stride;
  a.out = static_cast<uint16_t*>(grad_logits);
  a.ors = out_row_stride;
  a.M = M;
  a.V = V;
  a.targets = targets;
  a.tbytes = target_bytes;
  a.ignore = ignore_index;
  a.g = grad_loss;
  a.err = error_flag;
  if (want_loss) {
    a.row_loss = static_cast<double*>(workspace);
    a.row_valid = reinterpret_cast<int32_t*>(static_cast<char*>(workspace) + (size_t)M * sizeof(double));
  }
  if (M > 0) {
    // Rows in slabs of what one launch takes: its work-items and the targets'
    // buffer descriptor are 32-bit.
    const FbPlan plan = fb_plan(V);
    const int64_t by_blocks = plan.kernel != nullptr ? max_blocks(plan.threads) * plan.rows : max_blocks(kThreads);
    const int64_t slab = by_blocks < 0xffffffffLL / target_bytes ? by_blocks : 0xffffffffLL / target_bytes;
    for (int64_t r0 = 0; r0 < M; r0 += slab) {
      FbArgs b = a;
      b.M = M - r0 < slab ? M - r0 : slab;
      b.logits += r0 * row_stride;
      b.out += r0 * out_row_stride;
      b.targets = static_cast<const char*>(targets) + r0 * target_bytes;
      if (want_loss) {
        b.row_loss += r0;
        b.row_valid += r0;
      }
      void* args[] = {&b};
      if (plan.kernel != nullptr) {
        const int64_t cus = cu_count(), groups = ceil_div(b.M, plan.rows);
        const unsigned blocks = (unsigned)(plan.persistent && groups > cus ? cus : groups);
        launch_dominant_raw(reinterpret_cast<const void*>(plan.kernel), dim3(blocks), dim3(plan.threads), args, 0, st);
      } else {
        launch_dominant_raw(reinterpret_cast<const void*>(xent_fwd_bwd_scalar), dim3((unsigned)b.M), dim3(kThreads),
                            args, 0, st);
      }
      const int rc = check_launch(who);
      if (rc != KP_OK) return rc;
    }
  }
  if (!want_loss) return KP_OK;
  hipLaunchKernelGGL(xent_fwd_finish, dim3(1), dim3(kFinThreads), 0, st, a.row_loss, a.row_valid, M, (double)scale,
                     loss, total_weight);
  return check_launch(who);
}

}  // extern "C"
