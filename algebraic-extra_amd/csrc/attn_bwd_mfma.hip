// The MFMA attention backward for T a multiple of 128, and the dispatch
// between it and the kernels for any other T (attn_bwd_ragged.hip).
#define ALGX_ATTN_RAGGED 0
#include "attn_bwd_mfma_kernels.h"

namespace algx {

int32_t launch_bwd_mfma(const void* q, const void* k, const void* v, const float* stat,
                        const float* di, const void* dout, float* dq_acc, void* dk, void* dv,
                        int B, int H, int T, const KVariant& lo, const KVariant& hi,
                        const int32_t* guard, hipStream_t s) {
  auto fn = T % mfma::FBM == 0 ? mfma::launch_bwd_as : launch_bwd_ragged;
  return fn(q, k, v, stat, di, dout, dq_acc, dk, dv, B, H, T, lo, hi, guard, s);
}

}  // namespace algx
