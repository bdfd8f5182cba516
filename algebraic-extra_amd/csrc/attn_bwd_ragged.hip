// The MFMA attention backward for T that is no multiple of 128.
#define ALGX_ATTN_RAGGED 1
#include "attn_bwd_mfma_kernels.h"

namespace algx {

int32_t launch_bwd_ragged(const void* q, const void* k, const void* v, const float* stat,
                          const float* di, const void* dout, float* dq_acc, void* dk, void* dv,
                          int B, int H, int T, const KVariant& lo, const KVariant& hi,
                          const int32_t* guard, hipStream_t s) {
  return mfma::launch_bwd_as(q, k, v, stat, di, dout, dq_acc, dk, dv, B, H, T, lo, hi, guard, s);
}

}  // namespace algx
