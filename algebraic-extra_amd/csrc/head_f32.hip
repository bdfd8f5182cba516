// Fused head for float32 hidden states (fused_head.py:160-216 with h.dtype =
// float32: the embedding is cast to float32, the logits, their gradient dz and
// the products dh = dz E, dE = dz^T h are all float32).
//
// Every product runs on v_mfma_f32_32x32x2_f32 (float32 operands and sums): a
// 128 x 128 output tile per workgroup of 4 waves, 64 x 64 outputs each, 16-wide
// k stages double-buffered in LDS as [k][mn] and loaded one stage ahead through
// registers. Lane l = 32 g + c reads A[k + g][c] and B[k + g][c] and holds, in
// accumulator register r, row 8 (r / 4) + 4 g + r % 4 of column c. Bound by the
// matrix units: a stage is 2048 cycles of them per compute unit against 16 KB
// loaded and 64 KB of operand reads from LDS. N = 1024, d = 384, V = 32768,
// alg_ce, against 64 x 64 tiles of scalar FMAs (4 x 4 outputs a thread):
// forward 646 -> 301 us, dz 504 -> 282 us, dh and dE 6184 -> 574 + 8 us (dh had 96
// workgroups with a k loop over the whole vocabulary).
//
// Forward: grid (token tiles, vocabulary chunks); per-token online statistics
// merged over the lanes and waves that share a token and written as
// (chunk, token) partials for the head's statistics kernel. Backward: the logit
// gradient dz (float32, [tokens][V rounded up to 128]) of a token chunk, then
// the two products, each cut along k where its tiles alone would not fill the
// chip.
#include <initializer_list>

#include "head_f32.h"

namespace algx {
namespace {

constexpr int FT = 128;   // tile extent along m and n
constexpr int FK = 16;    // k stage
constexpr int FTHR = 256;
constexpr int FLD = FT + 4;  // LDS row stride (floats)
constexpr float kLog2eF = 1.4426950408889634f;
constexpr int kF32Groups = 512;  // workgroups that fill the chip (two per CU)

// C-tile operand: element (mn, k) at p[mn * s_mn + k * s_k], one of the strides
// 1, valid for mn < rows and k < K. VEC kernels read four consecutive elements
// at once where the first is valid: p 16-byte aligned, the other stride a
// multiple of 4, and what lies past a ragged end inside the allocation and
// without effect (dz's padding, outputs that are not stored).
struct F32Op {
  const float* p;
  int64_t s_mn, s_k;
  int rows, K;
};

__device__ __forceinline__ f32x16 mfma_f32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// One 128 x 16 stage of an operand in registers: two runs of 4 along the
// contiguous axis per thread.
template <bool VEC>
struct F32Stage {
  f32x4 v[2];
  static __device__ __forceinline__ void where(const F32Op& op, int e, int tid, int& mn, int& k) {
    const int id = tid + FTHR * e;
    if (op.s_k == 1) {
      mn = id / (FK / 4);
      k = id % (FK / 4) * 4;
    } else {
      k = id / (FT / 4);
      mn = id % (FT / 4) * 4;
    }
  }
  __device__ __forceinline__ void load(const F32Op& op, int mn0, int k0, int tid) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      int mn, k;
      where(op, e, tid, mn, k);
      mn += mn0;
      k += k0;
      if (VEC) {
        const bool in = mn < op.rows && k < op.K;
        const f32x4 x = *reinterpret_cast<const f32x4*>(
            op.p + (in ? (int64_t)mn * op.s_mn + (int64_t)k * op.s_k : 0));
#pragma unroll
        for (int u = 0; u < 4; ++u) v[e][u] = in ? x[u] : 0.0f;
      } else {
        const bool kc = op.s_k == 1;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int m = kc ? mn : mn + u, kk = kc ? k + u : k;
          v[e][u] = m < op.rows && kk < op.K
                        ? op.p[(int64_t)m * op.s_mn + (int64_t)kk * op.s_k] : 0.0f;
        }
      }
    }
  }
  __device__ __forceinline__ void store(const F32Op& op, float (*dst)[FLD], int tid) const {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      int mn, k;
      where(op, e, tid, mn, k);
      if (op.s_k == 1) {
#pragma unroll
        for (int u = 0; u < 4; ++u) dst[k + u][mn] = v[e][u];
      } else {
        *reinterpret_cast<f32x4*>(&dst[k][mn]) = v[e];
      }
    }
  }
};

struct F32Lds {
  float a[2][FK][FLD], b[2][FK][FLD];
};

// acc[i][j] of wave (wm, wn): rows m0 + 64 wm + 32 i + 8 (r / 4) + 4 g + r % 4,
// column n0 + 64 wn + 32 j + c, summed over the k stages [st0, st1).
template <bool VEC>
__device__ __forceinline__ void tile_f32(const F32Op& A, const F32Op& B, int m0, int n0, int st0,
                                         int st1, F32Lds& L, f32x16 (&acc)[2][2], int tid) {
  const int w = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int am = 64 * (w >> 1) + c, bn = 64 * (w & 1) + c;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  F32Stage<VEC> sa, sb;
  sa.load(A, m0, st0 * FK, tid);
  sb.load(B, n0, st0 * FK, tid);
  __syncthreads();  // the previous tile is no longer read
  sa.store(A, L.a[0], tid);
  sb.store(B, L.b[0], tid);
  __syncthreads();
  for (int st = st0; st < st1; ++st) {
    const int buf = (st - st0) & 1;
    if (st + 1 < st1) {
      sa.load(A, m0, (st + 1) * FK, tid);
      sb.load(B, n0, (st + 1) * FK, tid);
    }
#pragma unroll
    for (int k = 0; k < FK; k += 2) {
      float a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = L.a[buf][k + g][am + 32 * i];
        b[i] = L.b[buf][k + g][bn + 32 * i];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_f32(a[i], b[j], acc[i][j]);
    }
    if (st + 1 < st1) {
      sa.store(A, L.a[buf ^ 1], tid);
      sb.store(B, L.b[buf ^ 1], tid);
    }
    __syncthreads();
  }
}

__device__ __forceinline__ int stages_of(int K) { return (K + FK - 1) / FK; }

__device__ __forceinline__ float rho_fast_f(float x, float& r) {
  const float rad = __builtin_fmaf(x, x, 1.0f);
  r = rsq(rad);
  return __builtin_fmaf(rad, r, x);
}

// (m, l) <- the two states merged (ce), or the sums added (alg_ce).
template <int KIND>
__device__ __forceinline__ void merge_stat(float& m, float& l, float mo, float lo) {
  if (KIND == ALGX_HEAD_CE) {
    const float mm = __builtin_fmaxf(m, mo);
    l = l * __builtin_amdgcn_exp2f((m - mm) * kLog2eF) +
        lo * __builtin_amdgcn_exp2f((mo - mm) * kLog2eF);
    m = mm;
  } else {
    l += lo;
  }
}

// Forward statistics over one vocabulary chunk (fused_head.py:72-117),
// vocabulary rows on m, tokens on n.
// partial[(chunk * N + token) * 2 + {0, 1}] = (m, l) for ce, (0, l) for alg_ce.
template <int KIND, bool VEC>
__global__ __launch_bounds__(FTHR, 2) void head_f32_fwd_kernel(
    const float* __restrict__ h, const float* __restrict__ e, const int32_t* __restrict__ targets,
    float* __restrict__ zt, float* __restrict__ partial, int N, int d, int V, int log2n,
    float inv_c, float clamp, int chunk_tiles) {
  __shared__ F32Lds L;
  __shared__ float red_m[2][FT], red_l[2][FT];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int wm = w >> 1, wn = w & 1;
  const int n0 = blockIdx.x * FT, chunk = blockIdx.y;
  const int ntv = (V + FT - 1) / FT;
  const int t_begin = chunk * chunk_tiles;
  const int t_end = min(ntv, t_begin + chunk_tiles);
  const F32Op A{e, d, 1, V, d}, B{h, d, 1, N, d};
  float m_st[2], l_st[2];
  int tgt[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tok = n0 + 64 * wn + 32 * j + c;
    tgt[j] = tok < N ? targets[tok] : -1;
    m_st[j] = -1e30f;
    l_st[j] = 0.0f;
  }
  f32x16 acc[2][2];
  for (int t = t_begin; t < t_end; ++t) {
    const int m0 = t * FT;
    tile_f32<VEC>(A, B, m0, n0, 0, stages_of(d), L, acc, tid);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int tok = n0 + 64 * wn + 32 * j + c;
      float tmax = -1e30f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + 64 * wm + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
          if (m < V) {
            if (m == tgt[j]) zt[tok] = acc[i][j][r];
            if (KIND == ALGX_HEAD_CE) tmax = __builtin_fmaxf(tmax, acc[i][j][r]);
          }
        }
      const float m_new = __builtin_fmaxf(m_st[j], tmax);
      float lsum = 0.0f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + 64 * wm + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
          float wgt;
          if (KIND == ALGX_HEAD_CE) {
            wgt = __builtin_amdgcn_exp2f((acc[i][j][r] - m_new) * kLog2eF);
          } else {
            float rr;
            wgt = pow2n(rho_fast_f(__builtin_fminf(acc[i][j][r] * inv_c, clamp), rr), log2n);
          }
          lsum += m < V ? wgt : 0.0f;
        }
      if (KIND == ALGX_HEAD_CE) {
        l_st[j] = l_st[j] * __builtin_amdgcn_exp2f((m_st[j] - m_new) * kLog2eF) + lsum;
        m_st[j] = m_new;
      } else {
        l_st[j] += lsum;
      }
    }
  }
  // Merge the lane halves and the two waves that share a token.
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    merge_stat<KIND>(m_st[j], l_st[j], __shfl_xor(m_st[j], 32, 64), __shfl_xor(l_st[j], 32, 64));
    if (g == 0) {
      red_m[wm][64 * wn + 32 * j + c] = m_st[j];
      red_l[wm][64 * wn + 32 * j + c] = l_st[j];
    }
  }
  __syncthreads();
  if (tid < FT && n0 + tid < N) {
    float m = red_m[0][tid], l = red_l[0][tid];
    merge_stat<KIND>(m, l, red_m[1][tid], red_l[1][tid]);
    partial[((int64_t)chunk * N + n0 + tid) * 2 + 0] = KIND == ALGX_HEAD_CE ? m : 0.0f;
    partial[((int64_t)chunk * N + n0 + tid) * 2 + 1] = l;
  }
}

// dz[t][v] = f(z) * scale for the tokens [tok0, tok0 + ntok), 0 for v >= V
// (fused_head.py:127-145 with dz in float32). Tokens on m, vocabulary on n:
// 32 lanes store 32 consecutive columns.
template <int KIND, bool VEC>
__global__ __launch_bounds__(FTHR, 2) void head_f32_dz_kernel(
    const float* __restrict__ h, const float* __restrict__ e, const int32_t* __restrict__ targets,
    const float* __restrict__ stat, const float* __restrict__ scale, float* __restrict__ dz,
    int64_t ldz, int tok0, int ntok, int d, int V, int log2n, float inv_c, float clamp) {
  __shared__ F32Lds L;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int m0 = blockIdx.x * FT, n0 = blockIdx.y * FT;
  const F32Op A{h + (int64_t)tok0 * d, d, 1, ntok, d}, B{e, d, 1, V, d};
  f32x16 acc[2][2];
  tile_f32<VEC>(A, B, m0, n0, 0, stages_of(d), L, acc, tid);
  const float sc = scale[0];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int tl = m0 + 64 * (w >> 1) + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
      if (tl >= ntok) continue;
      const int tgt = targets[tok0 + tl];
      const float st = stat[tok0 + tl];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int v = n0 + 64 * (w & 1) + 32 * j + c;
        const float z = acc[i][j][r];
        const float y = v == tgt ? 1.0f : 0.0f;
        float gr;
        if (KIND == ALGX_HEAD_CE) {
          gr = __builtin_amdgcn_exp2f((z - st) * kLog2eF) - y;
        } else {
          float rr;
          const float p = pow2n(rho_fast_f(__builtin_fminf(z * inv_c, clamp), rr) * st, log2n);
          gr = (p - y) * rr;
        }
        dz[(int64_t)tl * ldz + v] = v < V ? gr * sc : 0.0f;
      }
    }
}

// C[m][n] (+)= sum_k A(m, k) B(n, k), C row-major with leading dimension ldc.
// gridDim.z > 1: chunk z sums the k stages [z * per, (z + 1) * per) into slice z
// of C (slices slice apart) instead.
template <bool VEC>
__global__ __launch_bounds__(FTHR, 2) void gemm_f32_kernel(F32Op A, F32Op B, float* __restrict__ C,
                                                           int64_t ldc, int64_t slice, int per,
                                                           int accumulate) {
  __shared__ F32Lds L;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 5, c = lane & 31;
  const int m0 = blockIdx.y * FT, n0 = blockIdx.x * FT;
  const int st0 = blockIdx.z * per, st1 = min(stages_of(A.K), st0 + per);
  f32x16 acc[2][2];
  tile_f32<VEC>(A, B, m0, n0, st0, st1, L, acc, tid);
  C += blockIdx.z * slice;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + 64 * (w >> 1) + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
      if (m >= A.rows) continue;
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = n0 + 64 * (w & 1) + 32 * j + c;
        if (n >= B.rows) continue;
        float* dst = C + (int64_t)m * ldc + n;
        *dst = accumulate ? *dst + acc[i][j][r] : acc[i][j][r];
      }
    }
}

// C (+)= the slices, added in chunk order.
__global__ __launch_bounds__(256) void gemm_f32_reduce(const float* __restrict__ P,
                                                       float* __restrict__ C, int64_t n, int splits,
                                                       int accumulate) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float s = P[i];
  for (int c = 1; c < splits; ++c) s += P[c * n + i];
  C[i] = accumulate ? C[i] + s : s;
}

// Vocabulary tiles per forward workgroup.
int chunk_tiles_f32(int N, int V) {
  const int nt = (V + FT - 1) / FT, ntb = (N + FT - 1) / FT;
  const int64_t per = ((int64_t)nt * ntb + kF32Groups - 1) / kF32Groups;
  return (int)(per < 1 ? 1 : per > nt ? nt : per);
}
int nchunks_f32(int N, int V) {
  const int nt = (V + FT - 1) / FT, ct = chunk_tiles_f32(N, V);
  return (nt + ct - 1) / ct;
}

int64_t vpad_f32(int V) { return ((int64_t)V + FT - 1) / FT * FT; }

// k chunks of a rows x cols product over K: enough workgroups to fill the chip,
// of 256 k or more each but the last, which takes what is left (a chunk's slice,
// written and read again, costs about what 64 k of its products do).
int gemm_splits(int rows, int cols, int K) {
  const int64_t tiles = (int64_t)((rows + FT - 1) / FT) * ((cols + FT - 1) / FT);
  int64_t s = tiles > 0 ? kF32Groups / tiles : 1;
  const int64_t cap = K / 256;
  if (s > cap) s = cap;
  return (int)(s < 1 ? 1 : s);
}
int64_t gemm_slice_bytes(int rows, int cols, int K) {
  const int s = gemm_splits(rows, cols, K);
  return s > 1 ? (int64_t)s * rows * cols * (int64_t)sizeof(float) : 0;
}

int32_t launch_gemm_f32(const F32Op& A, const F32Op& B, float* C, float* slices, bool vec,
                        bool accumulate, hipStream_t s) {
  if (A.rows == 0 || B.rows == 0) return 0;
  const int stages = (A.K + FK - 1) / FK, want = gemm_splits(A.rows, B.rows, A.K);
  const int per = (stages + want - 1) / want, splits = (stages + per - 1) / per;
  const int64_t n = (int64_t)A.rows * B.rows;
  dim3 grid((B.rows + FT - 1) / FT, (A.rows + FT - 1) / FT, splits);
  auto fn = vec ? gemm_f32_kernel<true> : gemm_f32_kernel<false>;
  const bool cut = splits > 1;
  fn<<<grid, FTHR, 0, s>>>(A, B, cut ? slices : C, (int64_t)B.rows, n, per,
                           !cut && accumulate ? 1 : 0);
  if (int32_t rc = check_launch("head_f32_gemm")) return rc;
  if (!cut) return 0;
  gemm_f32_reduce<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(slices, C, n, splits,
                                                             accumulate ? 1 : 0);
  return check_launch("head_f32_reduce");
}

// Four elements at a time: rows of h and E whole 16-byte pieces.
bool vec_ok(int d, const void* h, const void* E) {
  return d % 4 == 0 && ((uintptr_t)h & 15) == 0 && ((uintptr_t)E & 15) == 0;
}

}  // namespace

int64_t head_f32_fwd_workspace(int N, int V) { return (int64_t)nchunks_f32(N, V) * N * 2 * 4; }

int32_t head_f32_fwd(const float* h, const float* E, const int32_t* targets, float* zt,
                     float* partial, int N, int d, int V, int kind, int log2n, float inv_c,
                     float clamp, int* nchunks, hipStream_t s) {
  const int nch = nchunks_f32(N, V);
  *nchunks = nch;
  dim3 grid((N + FT - 1) / FT, nch);
  const bool vec = vec_ok(d, h, E);
  auto fn = kind == ALGX_HEAD_CE
                ? (vec ? head_f32_fwd_kernel<ALGX_HEAD_CE, true> : head_f32_fwd_kernel<ALGX_HEAD_CE, false>)
                : (vec ? head_f32_fwd_kernel<ALGX_HEAD_ALG_CE, true>
                       : head_f32_fwd_kernel<ALGX_HEAD_ALG_CE, false>);
  fn<<<grid, FTHR, 0, s>>>(h, E, targets, zt, partial, N, d, V, log2n, inv_c, clamp,
                           chunk_tiles_f32(N, V));
  return check_launch("head_f32_fwd");
}

// Tokens per backward chunk: the float32 dz scratch is capped at 2 GiB.
int head_f32_chunk_tokens(int N, int V) {
  const int64_t per_tok = vpad_f32(V) * 4;
  int64_t c = ((int64_t)2 << 30) / per_tok;
  c = c / FT * FT;
  if (c < FT) c = FT;
  return (int)(c > N ? N : c);
}

int64_t head_f32_bwd_workspace(int N, int d, int V) {
  const int csize = head_f32_chunk_tokens(N, V), last = N - (N - 1) / csize * csize;
  // the slices of either product, of a full chunk of tokens or the last one
  int64_t slices = 0;
  for (int ntok : {csize, last})
    for (int64_t b : {gemm_slice_bytes(ntok, d, V), gemm_slice_bytes(V, d, ntok)})
      slices = b > slices ? b : slices;
  return (int64_t)csize * vpad_f32(V) * 4 + slices;
}

int32_t head_f32_bwd(const float* h, const float* E, const int32_t* targets, const float* stat,
                     const float* scale, float* dh, float* dE, float* dz, int N, int d, int V,
                     int kind, int log2n, float inv_c, float clamp, hipStream_t s) {
  const int64_t ldz = vpad_f32(V);
  const int csize = head_f32_chunk_tokens(N, V);
  float* slices = dz + (int64_t)csize * ldz;
  const bool vec = vec_ok(d, h, E) && ((uintptr_t)dz & 15) == 0;
  auto zk = kind == ALGX_HEAD_CE
                ? (vec ? head_f32_dz_kernel<ALGX_HEAD_CE, true> : head_f32_dz_kernel<ALGX_HEAD_CE, false>)
                : (vec ? head_f32_dz_kernel<ALGX_HEAD_ALG_CE, true>
                       : head_f32_dz_kernel<ALGX_HEAD_ALG_CE, false>);
  for (int tok0 = 0; tok0 < N; tok0 += csize) {
    const int ntok = csize < N - tok0 ? csize : N - tok0;
    dim3 gdz((ntok + FT - 1) / FT, (V + FT - 1) / FT);
    zk<<<gdz, FTHR, 0, s>>>(h, E, targets, stat, scale, dz, ldz, tok0, ntok, d, V, log2n, inv_c,
                            clamp);
    if (int32_t rc = check_launch("head_f32_dz")) return rc;
    // dh[t][c] = sum_v dz[t][v] E[v][c]: A(m = t, k = v), B(n = c, k = v) = E[v][c].
    const F32Op adh{dz, ldz, 1, ntok, V}, bdh{E, 1, d, d, V};
    if (int32_t rc = launch_gemm_f32(adh, bdh, dh + (int64_t)tok0 * d, slices, vec, false, s))
      return rc;
    // dE[v][c] (+)= sum_t dz[t][v] h[t][c]: A(m = v, k = t), B(n = c, k = t) = h[t][c].
    const F32Op ade{dz, 1, ldz, V, ntok}, bde{h + (int64_t)tok0 * d, 1, d, d, ntok};
    if (int32_t rc = launch_gemm_f32(ade, bde, dE, slices, vec, tok0 > 0, s)) return rc;
  }
  return 0;
}

}  // namespace algx
