// One row of the bf16, D = 64 attention at a time, by a wave: a query's output
// or dq over its visible keys alone, a key's dk and dv over the queries that
// see it alone.
//
// The MFMA kernels give a masked key's or query's row the weight 0, and 0 times
// an infinity or NaN of that row is NaN. For T that is no multiple of 128 the
// kernels that came before skipped such rows, so these kernels form a row that
// came out non-finite again here: it is non-finite by its own inputs, or finite
// after all. Otherwise it costs a test of the results. A row all of whose values
// are NaN is left at once (inputs of NaN alone at B=8, H=16, T=2047: forward and
// backward 131 ms without that, 5.5 with). The callers mark the
// branch unlikely: by its loop depth alone the register allocator would spill
// the kernels' main loops for it.
#pragma once

#include "attn_common.h"

namespace algx {

// Lane l's products: row a (the same in all lanes, rounded to bf16 after a
// factor) with the lane's row b.
__device__ __forceinline__ float row_dot(const bf16* a, float factor, const bf16* b) {
  float s = 0.0f;
#pragma unroll 2
  for (int c = 0; c < 8; ++c) {
    const bf16x8 x = *reinterpret_cast<const bf16x8*>(a + 8 * c);
    const bf16x8 y = *reinterpret_cast<const bf16x8*>(b + 8 * c);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      s = __builtin_fmaf((float)(bf16)((float)x[e] * factor), (float)y[e], s);
  }
  return s;
}

// x of a lane (through LDS: a lane read by register may take its index from M0,
// which is the direct-to-LDS loads' alone).
__device__ __forceinline__ float from_lane(float x, int lane) { return __shfl(x, lane, 64); }

// acc += sum_j w(lane j) rows[j][lane], j < n.
__device__ __forceinline__ void row_add(float& acc, float w, const bf16* rows, int n, int lane) {
#pragma unroll 8
  for (int j = 0; j < n; ++j)
    acc = __builtin_fmaf(from_lane(w, j), (float)rows[j * 64 + lane], acc);
}

// Value `lane` of sum_j weight(score j) v_j over the keys j <= row of one head; q
// times factor is the pre-scaled query.
template <typename Weight>
__device__ __forceinline__ float row_forward(const bf16* q, float factor, const bf16* k,
                                             const bf16* v, int row, int lane, Weight&& weight) {
  float acc = 0.0f;
#pragma unroll 1
  for (int k0 = 0; k0 <= row; k0 += 64) {
    const int key = min(k0 + lane, row);
    const float p = weight(row_dot(q + (int64_t)row * 64, factor, k + (int64_t)key * 64));
    row_add(acc, (float)(bf16)p, v + (int64_t)k0 * 64, min(64, row - k0 + 1), lane);
    if (__all(acc != acc)) break;
  }
  return acc;
}

// p and ds of one score, rounded to bf16 (flash.py:339-361).
__device__ __forceinline__ void row_grad(const KVariant& var, float s, float dp, float st, float di,
                                         float& p, float& ds) {
  float rr;
  bool keep;
  p = bwd_weight(var, s, st, rr, keep);
  ds = p * (dp - di);
  if (var.kind == ALGX_ASINH) ds = keep ? ds * rr : 0.0f;
  p = (float)(bf16)p;
  ds = (float)(bf16)ds;
}

// Values `lane` of a key's dk (before the slope) and dv over the queries
// key .. T - 1 of one head.
__device__ __forceinline__ void row_dkdv(const KVariant& var, const bf16* q, const bf16* k,
                                         const bf16* v, const bf16* dout, const float* stat,
                                         const float* di, int key, int T, int lane, float& dk,
                                         float& dv) {
  dk = dv = 0.0f;
#pragma unroll 1
  for (int q0 = key; q0 < T; q0 += 64) {
    const int i = min(q0 + lane, T - 1), n = min(64, T - q0);
    const float s = row_dot(k + (int64_t)key * 64, 1.0f, q + (int64_t)i * 64);
    const float dp = row_dot(v + (int64_t)key * 64, 1.0f, dout + (int64_t)i * 64);
    float p, ds;
    row_grad(var, s, dp, stat[i], di[i], p, ds);
    row_add(dv, p, dout + (int64_t)q0 * 64, n, lane);
    row_add(dk, ds, q + (int64_t)q0 * 64, n, lane);
    if (__all(dk != dk && dv != dv)) break;
  }
}

// Value `lane` of a query's dq (before the slope) over the keys 0 .. row.
__device__ __forceinline__ float row_dq(const KVariant& var, const bf16* q, const bf16* k,
                                        const bf16* v, const bf16* dout, float stat, float di,
                                        int row, int lane) {
  float acc = 0.0f;
#pragma unroll 1
  for (int k0 = 0; k0 <= row; k0 += 64) {
    const int key = min(k0 + lane, row);
    const float s = row_dot(q + (int64_t)row * 64, 1.0f, k + (int64_t)key * 64);
    const float dp = row_dot(dout + (int64_t)row * 64, 1.0f, v + (int64_t)key * 64);
    float p, ds;
    row_grad(var, s, dp, stat, di, p, ds);
    row_add(acc, ds, k + (int64_t)k0 * 64, min(64, row - k0 + 1), lane);
    if (__all(acc != acc)) break;
  }
  return acc;
}

}  // namespace algx
