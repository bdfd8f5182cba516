// The MFMA attention forward for T in whole 128-query blocks, and the
// dispatch between it and the kernels for any other T (attn_fwd_ragged.hip).
#define ALGX_ATTN_RAGGED 0
#include "attn_fwd_mfma_kernels.h"

namespace algx {

bool mfma_supported(int T, int D, int dtype) {
  return dtype == ALGX_BF16 && D == mfma::HD && T > 0;
}

bool mfma_pair(const KVariant& lo, const KVariant& hi) {
  return mfma::pair_ok(mfma::cfg_for(lo), mfma::cfg_for(hi));
}

bool mfma_fused_pair(const KVariant&, const KVariant& hi) {
  return mfma::high_ok(mfma::cfg_for(hi));
}

int64_t fwd_fused_partials(int B, int H, int T) {
  return (int64_t)B * H * ((T + mfma::FBM - 1) / mfma::FBM);
}

int32_t launch_fwd_mfma(const void* q, const void* k, const void* v, const float* sink, void* o,
                        float* o_precise, float* stat, int B, int H, int T, const KVariant& lo,
                        const KVariant& hi, const int32_t* guard, hipStream_t s) {
  auto fn = T % mfma::FBM == 0 ? mfma::launch_fwd_as : launch_fwd_ragged;
  return fn(q, k, v, sink, o, o_precise, stat, B, H, T, lo, hi, guard, s);
}

int32_t launch_fwd_fused(const void* q, const void* k, const void* v, const float* sink,
                         void* q_s, void* o, float* o_precise, float* stat, int32_t* guard,
                         float* partial, float* dq_zero, int B, int H, int T, float q_scale,
                         float bound, float vmax, const KVariant& lo, const KVariant& hi,
                         hipStream_t s) {
  auto fn = T % mfma::FBM == 0 ? mfma::launch_fused_as : launch_fused_ragged;
  return fn(q, k, v, sink, q_s, o, o_precise, stat, guard, partial, dq_zero, B, H, T, q_scale,
            bound, vmax, lo, hi, s);
}

}  // namespace algx
