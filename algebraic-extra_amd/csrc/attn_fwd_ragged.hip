// The MFMA attention forward for T that is no multiple of 128.
#define ALGX_ATTN_RAGGED 1
#include "attn_fwd_mfma_kernels.h"

namespace algx {

int32_t launch_fwd_ragged(const void* q, const void* k, const void* v, const float* sink, void* o,
                          float* o_precise, float* stat, int B, int H, int T, const KVariant& lo,
                          const KVariant& hi, const int32_t* guard, hipStream_t s) {
  return mfma::launch_fwd_as(q, k, v, sink, o, o_precise, stat, B, H, T, lo, hi, guard, s);
}

int32_t launch_fused_ragged(const void* q, const void* k, const void* v, const float* sink,
                            void* q_s, void* o, float* o_precise, float* stat, int32_t* guard,
                            float* partial, float* dq_zero, int B, int H, int T, float q_scale,
                            float bound, float vmax, const KVariant& lo, const KVariant& hi,
                            hipStream_t s) {
  return mfma::launch_fused_as(q, k, v, sink, q_s, o, o_precise, stat, guard, partial, dq_zero, B,
                               H, T, q_scale, bound, vmax, lo, hi, s);
}

}  // namespace algx
