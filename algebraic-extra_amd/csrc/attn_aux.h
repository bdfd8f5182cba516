// Host-side launchers shared by the attention entry points.
#pragma once

#include "attn_common.h"

namespace algx {

int32_t guard_words();
// q_s = cast(q * q_scale); with a guard buffer also the range-guard word.
int32_t launch_prepare(const void* q, const void* k, const void* v, const float* sink, void* q_s,
                       int32_t* guard, int B, int H, int T, int D, int dtype, float q_scale,
                       float bound, float vmax, float sink_unit, hipStream_t s);
// Guard word from `nblocks` triples of partial maxima (|q_s|^2, |k|^2, |v|).
int32_t launch_guard_finish(const float* partial, int nblocks, const float* sink, int H,
                            float bound, float vmax, float sink_unit, int32_t* guard,
                            hipStream_t s);
// The sink gradient's shares of the backward pre-pass (nblk per (b, h)) and
// where their sums go; dsink null: no sink gradient.
struct SinkGrad {
  const float* part;
  float* dsink;
  int nblk, B, H;
  float unit;  // the sink's
};
// Row pre-pass of the backward: di (and, with a sink and sink_part, each
// block's share of the sink gradient, pre_blocks() per (b, h)), and the dQ
// accumulator (T in whole 128-row blocks) cleared when dq_acc is given.
int pre_blocks(int T, int D, int dtype);
int32_t launch_bwd_pre(const void* dout, const void* o, const float* o_precise,
                       const float* stat, const float* sink, float* di, float* dq_acc,
                       float* sink_part, int B, int H, int T, int D, int dtype,
                       const KVariant& low, const KVariant& high, const int32_t* guard,
                       hipStream_t s);
// dsink from the shares, as a launch of its own or in the dQ finish.
int32_t launch_sink_finish(const SinkGrad& sg, hipStream_t s);
// dq (bf16, D = 64) of the MFMA backward from its float32 sums.
struct BwdRows {  // what the backward read, for rows formed again (attn_rows.h)
  const bf16 *q, *k, *v, *dout;
  const float *stat, *di;
};
int32_t launch_dq_finish(const float* acc, void* dq, const BwdRows& in, int B, int H, int T,
                         const KVariant& low, const KVariant& high, const int32_t* guard,
                         float q_scale, const SinkGrad& sg, hipStream_t s);

// Generic kernels: any T, D in {16, 32, 64}, bf16 or f32, every variant. With a
// guard word they run `lo` or `hi` for the whole call, else `lo`.
int32_t launch_fwd_generic(const void* q_s, const void* k, const void* v, const float* sink,
                           void* o, float* o_precise, float* stat, int B, int H, int T, int D,
                           int dtype, const KVariant& lo, const KVariant& hi, const int32_t* guard,
                           hipStream_t s);
int32_t launch_bwd_generic(const void* q, const void* k, const void* v, const float* stat,
                           const float* di, const void* dout, void* dq, void* dk, void* dv,
                           int B, int H, int T, int D, int dtype, float q_scale,
                           const KVariant& lo, const KVariant& hi, const int32_t* guard,
                           hipStream_t s);

// MFMA kernels: bf16, D = 64, any T.
bool mfma_supported(int T, int D, int dtype);
// Whether they have the variant pair of a guarded call: one launch for both
// (algx_attn_fwd, the backward), or the fused forward's two. Without it the
// generic kernels run at T that is no multiple of 128, as for any variants
// there; other T have no other kernels and are refused.
bool mfma_pair(const KVariant& lo, const KVariant& hi);
bool mfma_fused_pair(const KVariant& lo, const KVariant& hi);
// Rows per head of the MFMA backward's float32 dQ sums: T rounded up to whole
// 128-row query blocks, so that the backward stores whole tiles.
__host__ __device__ inline int acc_rows(int T) { return (T + 127) / 128 * 128; }
// Keys of a workgroup of the MFMA backward.
constexpr int kBwdKeys = 256;
// Copies (slots) of those sums in the workspace. One where T is a multiple of
// 128: the key blocks add to it with atomics. Elsewhere dq is the same in every
// run, as it was on the generic kernels: a launch takes at most this many key
// blocks, each with a slot of its own, the next launch adds its blocks to the
// slots, and the finish adds the slots in order. Four at least, else as many as
// one launch of a workgroup per compute unit takes, so that the slots of a
// large batch stay at four. The reads of the finish are the price: all kernels
// of a guarded forward and backward, against atomics into one accumulator (and
// di as two bf16 values, no row formed again), B=2, H=12, T=333 54.1 -> 53.2 us,
// B=8, H=16, T=700 99.8 -> 97.5, B=8, H=24, T=1023 225 -> 239 (finish 13 -> 25),
// B=8, H=16, T=2047 444 -> 477 us (finish 17 -> 39, backward 289 -> 302).
inline int dq_slots(int B, int H, int T, int D) {
  const int64_t bh = (int64_t)B * H;
  if (D != 64 || T % 128 == 0 || bh <= 0) return 1;
  const int64_t nkb = (T + kBwdKeys - 1) / kBwdKeys, fill = (256 + bh - 1) / bh;
  const int64_t n = fill > 4 ? fill : 4;
  return (int)(n < nkb ? n : nkb);
}
// One launch per call: with a guard word the kernel runs `lo` or `hi` for the
// whole grid; without one it runs `lo`.
int32_t launch_fwd_mfma(const void* q_s, const void* k, const void* v, const float* sink,
                        void* o, float* o_precise, float* stat, int B, int H, int T,
                        const KVariant& lo, const KVariant& hi, const int32_t* guard,
                        hipStream_t s);
// Pre-scale, guard and forward in one pass over q (MFMA shapes): the low
// variant runs over the whole grid writing q_s and, guarded, one triple of
// partial maxima per workgroup (fwd_fused_partials of them); a second launch
// reduces them to the guard word and, out of range only, runs the high
// variant. dq_zero (or null): the backward's dQ accumulator, cleared in the
// same pass.
int64_t fwd_fused_partials(int B, int H, int T);
int32_t launch_fwd_fused(const void* q, const void* k, const void* v, const float* sink,
                         void* q_s, void* o, float* o_precise, float* stat, int32_t* guard,
                         float* partial, float* dq_zero, int B, int H, int T, float q_scale,
                         float bound, float vmax, const KVariant& lo, const KVariant& hi,
                         hipStream_t s);
int32_t launch_bwd_mfma(const void* q_s, const void* k, const void* v, const float* stat,
                        const float* di, const void* dout, float* dq_acc, void* dk, void* dv,
                        int B, int H, int T, const KVariant& lo, const KVariant& hi,
                        const int32_t* guard, hipStream_t s);

// The same launches for T that is no multiple of 128 (translation units of
// their own).
int32_t launch_fwd_ragged(const void* q_s, const void* k, const void* v, const float* sink,
                          void* o, float* o_precise, float* stat, int B, int H, int T,
                          const KVariant& lo, const KVariant& hi, const int32_t* guard,
                          hipStream_t s);
int32_t launch_fused_ragged(const void* q, const void* k, const void* v, const float* sink,
                            void* q_s, void* o, float* o_precise, float* stat, int32_t* guard,
                            float* partial, float* dq_zero, int B, int H, int T, float q_scale,
                            float bound, float vmax, const KVariant& lo, const KVariant& hi,
                            hipStream_t s);
int32_t launch_bwd_ragged(const void* q, const void* k, const void* v, const float* stat,
                          const float* di, const void* dout, float* dq_acc, void* dk, void* dv,
                          int B, int H, int T, const KVariant& lo, const KVariant& hi,
                          const int32_t* guard, hipStream_t s);

}  // namespace algx
