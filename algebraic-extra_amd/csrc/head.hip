// Fused tied-embedding projection + likelihood loss (fused_head.py) on gfx950.
//
// Forward (fused_head.py:72-117, :174-191): logits z^T = E h^T are formed
// tile by tile (256 vocab x 256 tokens, d streamed through LDS in 32-wide
// stages, v_mfma_f32_32x32x16_bf16) and never stored. Vocabulary rows sit on
// the MFMA M axis so every lane holds 16 vocabulary values of one token; the
// per-token statistic (online max/sum-exp for "ce", sum of rho(min(z/c,X))^n
// for "alg_ce") is kept per lane, merged across lanes at the end of a
// workgroup's vocabulary chunk, and merged across chunks by a small kernel.
// The target logit is written by the one lane that meets it.
//
// Backward (fused_head.py:120-156, :194-216): the same tiles are recomputed
// and the scaled bf16 logit gradient dz (fused_head.py:145) is written for a
// chunk of tokens; dh = dz E and dE += dz^T h are then plain MFMA GEMMs over
// that chunk (the reference also materialises dz and runs an XLA GEMM for dE).
#include <cstdlib>
#include <type_traits>

#include "gemm_core.h"
#include "head_f32.h"

namespace algx {

namespace {

constexpr int kFwdWorkgroups = 256;  // forward grid target: one workgroup per CU

// x^n, n = 2^log2n: unrolled squarings for a compile-time L2N > 0 (a runtime
// loop inside the per-logit epilogue would cost a branch per logit).
template <int L2N> __device__ __forceinline__ float pow_n(float x, int log2n) {
  if (L2N > 0) {
#pragma unroll
    for (int i = 0; i < L2N; ++i) x = x * x;
    return x;
  }
  return pow2n(x, log2n);
}

// alg_ce weight w = (x + sqrt(1+x^2))^n with x = min(z/c, clamp) (fused_head.py:98-100).
template <int L2N>
__device__ __forceinline__ float alg_weight(float z, float inv_c, float clamp, int log2n,
                                            float& r) {
  const float x = __builtin_fminf(z * inv_c, clamp);
  return pow_n<L2N>(rho_fast(x, r), log2n);
}

// Forward statistics. grid = (token blocks) x (vocabulary chunks of
// chunk_tiles tiles).
// partial[(chunk * N + token) * 2 + {0,1}] = (m, l) for ce, (-, l) for alg_ce.
// DMA: the direct-to-LDS ring streamed over the chunk's tiles (d a multiple
// of BK * kDmaStages).
template <int KIND, int L2N, bool DMA>
__global__ __launch_bounds__(kThreads) void head_fwd_kernel(
    const bf16* __restrict__ h, const bf16* __restrict__ e, const int32_t* __restrict__ targets,
    float* __restrict__ zt, float* __restrict__ partial, int N, int d, int V, int log2n,
    float inv_c, float clamp, int chunk_tiles) {
  GEMM_LDS_STAGES;
  __shared__ float red_m[2][BN], red_l[2][BN];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 5, c32 = lane & 31;
  const int wm = w / NWN, wn = w % NWN;
  const int n0 = blockIdx.x * BN;
  const int chunk = blockIdx.y;
  const int ntiles_v = (V + BM - 1) / BM;
  const int t_begin = chunk * chunk_tiles;
  const int t_end = min(ntiles_v, t_begin + chunk_tiles);
  const Operand A{e, d, V, d};
  const Operand B{h, d, N, d};
  int tok[TJ], tgt[TJ];
  float m_st[TJ], l_st[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    tok[j] = n0 + WTN * wn + 32 * j + c32;
    tgt[j] = tok[j] < N ? targets[tok[j]] : -1;
    m_st[j] = -1e30f;
    l_st[j] = 0.0f;
  }
  // Statistic update of one vocabulary tile; FULL: every row of the tile is
  // inside the vocabulary (all but the last tile), so no row mask is formed.
  auto consume = [&](auto full_tag, int m0, const Acc& acc) {
    constexpr bool FULL = decltype(full_tag)::value;
    const int mw = m0 + WTM * wm;
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      // The target logit: one lane of one 32-row block holds it. The wave's
      // 128 rows hold a target of its 32 tokens in ~8 % of the (tile,
      // column) pairs at V = 50304, so one wave-wide vote skips the search.
      if (__any((unsigned)(tgt[j] - mw) < (unsigned)WTM)) {
#pragma unroll
        for (int i = 0; i < TI; ++i) {
          const int off = tgt[j] - (mw + 32 * i);
          if (off >= 0 && off < 32 && ((off >> 2) & 1) == g) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
              if (8 * (r >> 2) + (r & 3) == (off & ~4)) zt[tok[j]] = acc.v[i][j][r];
          }
        }
      }
      float tile_max = -1e30f;
      if (KIND == ALGX_HEAD_CE) {
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int m = mw + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
            if (FULL || m < V) tile_max = __builtin_fmaxf(tile_max, acc.v[i][j][r]);
          }
      }
      const float m_new = __builtin_fmaxf(m_st[j], tile_max);
      float lsum = 0.0f;
#pragma unroll
      for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mw + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
          const float z = acc.v[i][j][r];
          float wgt;
          if (KIND == ALGX_HEAD_CE) {
            wgt = __builtin_amdgcn_exp2f((z - m_new) * 1.4426950408889634f);
          } else {
            float rr;
            wgt = alg_weight<L2N>(z, inv_c, clamp, log2n, rr);
          }
          lsum += (FULL || m < V) ? wgt : 0.0f;
        }
      if (KIND == ALGX_HEAD_CE) {
        l_st[j] = l_st[j] * __builtin_amdgcn_exp2f((m_st[j] - m_new) * 1.4426950408889634f) + lsum;
        m_st[j] = m_new;
      } else {
        l_st[j] += lsum;
      }
    }
  };
  Acc acc;
  if constexpr (DMA) {
    gemm_seq_dma<true, true>(A, B, t_begin * BM, t_end - t_begin, n0, ring, acc, tid,
                             [&](int, int m0, const Acc& a) {
                               if (m0 + BM <= V)
                                 consume(std::true_type{}, m0, a);
                               else
                                 consume(std::false_type{}, m0, a);
                             });
  } else {
    for (int t = t_begin; t < t_end; ++t) {
      const int m0 = t * BM;
      gemm_tile<true, true>(A, B, m0, n0, s0, s0 + 2 * kStageElems, acc, tid);
      if (m0 + BM <= V)
        consume(std::true_type{}, m0, acc);
      else
        consume(std::false_type{}, m0, acc);
    }
  }
  // Merge the 4 partial states of each token: lane halves g, then waves wm.
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    float mo = __shfl_xor(m_st[j], 32, 64), lo = __shfl_xor(l_st[j], 32, 64);
    if (KIND == ALGX_HEAD_CE) {
      const float mm = __builtin_fmaxf(m_st[j], mo);
      l_st[j] = l_st[j] * __builtin_amdgcn_exp2f((m_st[j] - mm) * 1.4426950408889634f) +
                lo * __builtin_amdgcn_exp2f((mo - mm) * 1.4426950408889634f);
      m_st[j] = mm;
    } else {
      l_st[j] += lo;
    }
    if (g == 0) {
      red_m[wm][WTN * wn + 32 * j + c32] = m_st[j];
      red_l[wm][WTN * wn + 32 * j + c32] = l_st[j];
    }
  }
  __syncthreads();
  if (tid < BN) {
    const int col = tid;
    const float m_a = red_m[0][col], l_a = red_l[0][col];
    const float m_b = red_m[1][col], l_b = red_l[1][col];
    float m_out, l_out;
    if (KIND == ALGX_HEAD_CE) {
      m_out = __builtin_fmaxf(m_a, m_b);
      l_out = l_a * __builtin_amdgcn_exp2f((m_a - m_out) * 1.4426950408889634f) +
              l_b * __builtin_amdgcn_exp2f((m_b - m_out) * 1.4426950408889634f);
    } else {
      m_out = 0.0f;
      l_out = l_a + l_b;
    }
    const int token = n0 + col;
    if (token < N) {
      partial[((int64_t)chunk * N + token) * 2 + 0] = m_out;
      partial[((int64_t)chunk * N + token) * 2 + 1] = l_out;
    }
  }
}

// What the chunk partials of a token become. stat = m + log l (ce) or
// l^(-1/n) (alg_ce) (fused_head.py:113-116); with tel, also the per-token NLL
// or target probability and the block's share of the objective
// (fused_head.py:219-229).
struct HeadStat {
  const float* partial;
  const int32_t* targets;
  float* zt;        // target logits; a target outside the vocabulary reads 0
  float* stat;
  float* tel;       // null: stat and zt only
  float* obj_part;  // one share per block
  int nchunks, N, V, log2n;
  float inv_c, clamp;
};

// A workgroup takes 64 tokens, its four waves every fourth chunk each: few
// tokens come with many chunks, and one thread per token walked them serially
// on a handful of CUs (18 us at N = 1024 with 64 chunks, now 4.5 us).
constexpr int kStatTokens = 64;

template <int KIND>
__global__ __launch_bounds__(256) void head_stat_kernel(HeadStat p) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  constexpr float kLog2e = 1.4426950408889634f;
  __shared__ float red_m[4][kStatTokens], red_l[4][kStatTokens];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x * kStatTokens + lane;
  float m = -1e30f, l = 0.0f;
  auto merge = [&](float mo, float lo) {
    if (KIND == ALGX_HEAD_CE) {
      const float mm = __builtin_fmaxf(m, mo);
      l = l * __builtin_amdgcn_exp2f((m - mm) * kLog2e) +
          lo * __builtin_amdgcn_exp2f((mo - mm) * kLog2e);
      m = mm;
    } else {
      l += lo;
    }
  };
  if (t < p.N) {
#pragma unroll 4
    for (int c = w; c < p.nchunks; c += 4) {
      const f32x2 x = *reinterpret_cast<const f32x2*>(p.partial + ((int64_t)c * p.N + t) * 2);
      merge(x[0], x[1]);
    }
  }
  red_m[w][lane] = m;
  red_l[w][lane] = l;
  __syncthreads();
  if (w != 0) return;
#pragma unroll
  for (int ww = 1; ww < 4; ++ww) merge(red_m[ww][lane], red_l[ww][lane]);
  float term = 0.0f;
  if (t < p.N) {
    const float st = KIND == ALGX_HEAD_CE ? m + __logf(l) : inv_root(l, p.log2n);
    p.stat[t] = st;
    const int tgt = p.targets[t];
    float z = 0.0f;
    if ((unsigned)tgt < (unsigned)p.V)
      z = p.zt[t];
    else
      p.zt[t] = 0.0f;
    if (p.tel != nullptr) {
      float tel;
      if (KIND == ALGX_HEAD_CE) {
        tel = st - z;
        term = tel;
      } else {
        // A comparison, not a minimum: a NaN logit stays NaN, and so do the
        // objective and a trainer's check of it. -inf becomes NaN (x - x), as
        // the same expression on materialised logits gives.
        float x = z * p.inv_c;
        x = x > p.clamp ? p.clamp : x;
        const float r = __builtin_fabsf(x) + __builtin_sqrtf(__builtin_fmaf(x, x, 1.0f));
        tel = pow2n((x >= 0.0f ? r : 1.0f / r) * st, p.log2n) + (x - x);
        term = 1.0f - tel;
      }
      p.tel[t] = tel;
    }
  }
  if (p.tel == nullptr) return;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) term += __shfl_xor(term, s, 64);
  if (lane == 0) p.obj_part[blockIdx.x] = term;
}

// obj = the mean over the tokens from the blocks' shares.
__global__ __launch_bounds__(256) void head_mean_kernel(const float* __restrict__ part, int nparts,
                                                        int N, float* __restrict__ obj) {
  __shared__ float red[4];
  float s = 0.0f;
  for (int i = threadIdx.x; i < nparts; i += 256) s += part[i];
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) s += __shfl_xor(s, m, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) obj[0] = ((red[0] + red[1]) + (red[2] + red[3])) / (float)N;
}

// dz tile of a token chunk: dz[t][v] = bf16(f(z) * scale), 0 for padded v.
// BLK = false: dz row-major with row stride ldz. BLK: dz is stored in blocks
// of 32 vocabulary columns, [v / 32][t][32] with blocks bstride apart (the
// layout the backward's GEMMs read in whole 64-byte row pieces).
template <int KIND, int L2N, bool DMA, bool BLK>
__global__ __launch_bounds__(kThreads) void head_dz_kernel(
    const bf16* __restrict__ h, const bf16* __restrict__ e, const int32_t* __restrict__ targets,
    const float* __restrict__ stat, const float* __restrict__ scale, bf16* __restrict__ dz,
    int64_t ldz, int64_t bstride, int tok0, int ntok, int d, int V, int log2n, float inv_c,
    float clamp, int chunk_tiles) {
  GEMM_LDS_STAGES;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, g = lane >> 5, c32 = lane & 31;
  const int wm = w / NWN, wn = w % NWN;
  const int n0 = blockIdx.x * BN;  // token offset inside the chunk
  const int ntiles_v = (V + BM - 1) / BM;
  const int t_begin = blockIdx.y * chunk_tiles;
  const int t_end = min(ntiles_v, t_begin + chunk_tiles);
  const Operand A{e, d, V, d};
  const Operand B{h + (int64_t)tok0 * d, d, ntok, d};
  // The lane's tokens (the same for every vocabulary tile), read before the
  // loads of the stage ring start.
  int tgt_j[TJ];
  float st_j[TJ];
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int tl = n0 + WTN * wn + 32 * j + c32;
    tgt_j[j] = tl < ntok ? targets[tok0 + tl] : -1;
    st_j[j] = tl < ntok ? stat[tok0 + tl] : 0.0f;
  }
  const float sc = scale[0];
  // FULL: every row of the tile is inside the vocabulary (all but the last
  // vocabulary tile), so no row mask is formed.
  auto emit = [&](auto full_tag, int m0, const Acc& acc) {
    constexpr bool FULL = decltype(full_tag)::value;
    // dz of columns mb0 + 8 q4 + 4 g .. + 3 of token column j
    // d loss / d z of one logit, y the target indicator (fused_head.py:137-145)
    auto grad = [&](float z, float y, float st) {
      if (KIND == ALGX_HEAD_CE)
        return __builtin_amdgcn_exp2f((z - st) * 1.4426950408889634f) - y;
      const float x = __builtin_fminf(z * inv_c, clamp);
      float r;
      const float p = pow_n<L2N>(rho_fast(x, r) * st, log2n);
      return (p - y) * r;
    };
    // TGT: some lane of the wave has its token's target among the rows it
    // holds for this token column, so each logit takes the indicator y; else
    // y = 0 everywhere ((p - 0) r = p r exactly, so both forms agree bitwise).
    auto run = [&](auto tgt_tag, int mb0, int i, int j, int q4, int tgt, float st) {
      constexpr bool TGT = decltype(tgt_tag)::value;
      bf16x4 out;
      const int mr = mb0 + 8 * q4 + 4 * g;  // the run's first column
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float y = TGT && mr + u == tgt ? 1.0f : 0.0f;
        out[u] = (bf16)((FULL || mr + u < V) ? grad(acc.v[i][j][4 * q4 + u], y, st) * sc : 0.0f);
      }
      return out;
    };
    auto column = [&](auto tgt_tag, int j) {
      const int tl = n0 + WTN * wn + 32 * j + c32;  // the same in lanes c32 and c32 + 32
      const int tgt = tgt_j[j];
      const float st = st_j[j];
#pragma unroll
      for (int i = 0; i < TI; ++i) {
        const int mb0 = m0 + WTM * wm + 32 * i;  // a 32-column block of dz
        if (tl >= ntok) continue;  // both lanes of a swap pair
        if constexpr (BLK) {
          // Lanes c32 and c32 + 32 hold alternate 4-column runs of one
          // token's 32 columns. Per pair of runs, two swaps between the lane
          // halves give each lane 8 consecutive columns, stored as 16 bytes:
          // columns 16 h + 8 g .. + 7 of the block.
          bf16* row = dz + (int64_t)(mb0 >> 5) * bstride + (int64_t)tl * 32 + 8 * g;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            u32x2 d0 = __builtin_bit_cast(u32x2, run(tgt_tag, mb0, i, j, 2 * h, tgt, st));
            u32x2 d1 = __builtin_bit_cast(u32x2, run(tgt_tag, mb0, i, j, 2 * h + 1, tgt, st));
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              // upper half of d0[e] <-> lower half of d1[e]
              const auto r = __builtin_amdgcn_permlane32_swap(d0[e], d1[e], false, false);
              d0[e] = r[0];
              d1[e] = r[1];
            }
            *reinterpret_cast<u32x4*>(row + 16 * h) = u32x4{d0[0], d0[1], d1[0], d1[1]};
          }
        } else {
#pragma unroll
          for (int q4 = 0; q4 < 4; ++q4)
            *reinterpret_cast<bf16x4*>(dz + (int64_t)tl * ldz + mb0 + 8 * q4 + 4 * g) =
                run(tgt_tag, mb0, i, j, q4, tgt, st);
        }
      }
    };
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
      // A wave's 128 rows hold a target of its 32 tokens in ~8 % of the
      // (tile, column) pairs at V = 50304; the test is one wave-wide vote.
      const bool hit = (unsigned)(tgt_j[j] - (m0 + WTM * wm)) < (unsigned)WTM;
      if (__any(hit))
        column(std::true_type{}, j);
      else
        column(std::false_type{}, j);
    }
  };
  auto emit_tile = [&](int, int m0, const Acc& a) {
    if (m0 + BM <= V)
      emit(std::true_type{}, m0, a);
    else
      emit(std::false_type{}, m0, a);
  };
  Acc acc;
  if constexpr (DMA) {
    gemm_seq_dma<true, true, true>(A, B, t_begin * BM, t_end - t_begin, n0, ring, acc, tid,
                                   emit_tile);
  } else {
    for (int t = t_begin; t < t_end; ++t) {
      gemm_tile<true, true>(A, B, t * BM, n0, s0, s0 + 2 * kStageElems, acc, tid);
      emit_tile(t, t * BM, acc);
    }
  }
}

// One GEMM of a grouped launch: C[m][n] (+)= sum_k A(m,k) B(n,k).
struct GemmJob {
  Operand A, B;
  void* C;
  int64_t ldc;
  int M, N;
  int tiles_n;  // output tiles along n
};

// acc of tile (m0, n0) into C; v(i, j, r) gives its values.
template <typename TOut, bool ACCUM, typename Val>
__device__ __forceinline__ void put_tile(const GemmJob& jb, int m0, int n0, int i, int j, int tid,
                                         Val&& v) {
  const int w = tid >> 6, lane = tid & 63, g = lane >> 5, c32 = lane & 31;
  const int wm = w / NWN, wn = w % NWN;
  const int n = n0 + WTN * wn + 32 * j + c32;
  if (n >= jb.N) return;
  TOut* C = reinterpret_cast<TOut*>(jb.C);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + WTM * wm + 32 * i + 8 * (r >> 2) + 4 * g + (r & 3);
    if (m >= jb.M) continue;
    TOut* dst = C + (int64_t)m * jb.ldc + n;
    if (ACCUM)
      *dst = from_f<TOut>(to_f(*dst) + v(r));
    else
      *dst = from_f<TOut>(v(r));
  }
}

// A unit's float32 sums of a tile in the workspace, in the accumulators'
// order: run q (4 values) of block (i, j) of thread tid is one 16-byte piece.
constexpr int kSlotElems = BM * BN;
__device__ __forceinline__ int64_t slot_at(int i, int j, int q, int tid) {
  return ((int64_t)((i * TJ + j) * 4 + q) * kThreads + tid) * 4;
}

// K stages [st0, st1) of one output tile; slot null: written to C, else the
// float32 sums go to the slot.
template <bool AKC, bool BKC, typename TOut, bool ACCUM, bool DMA>
__device__ __forceinline__ void gemm_job(const GemmJob& jb, int tile, int st0, int st1,
                                         float* slot, bf16* lds, const DmaRing& ring, int tid) {
  const int m0 = (tile / jb.tiles_n) * BM, n0 = (tile % jb.tiles_n) * BN;
  Acc acc;
  if (DMA)
    gemm_tile_range<AKC, BKC>(jb.A, jb.B, m0, n0, st0, st1, ring, acc, tid);
  else
    gemm_tile<AKC, BKC>(jb.A, jb.B, m0, n0, lds, lds + 2 * kStageElems, acc, tid);
  if (DMA && slot != nullptr) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<f32x4*>(slot + slot_at(i, j, q, tid)) =
              f32x4{acc.v[i][j][4 * q], acc.v[i][j][4 * q + 1], acc.v[i][j][4 * q + 2],
                    acc.v[i][j][4 * q + 3]};
    return;
  }
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      put_tile<TOut, ACCUM>(jb, m0, n0, i, j, tid, [&](int r) { return acc.v[i][j][r]; });
}

// How the backward's two products are dealt to workgroups (grad_plan): every
// dh tile in s1 chunks of c1 k stages, the first n_de - n_tail dE tiles whole
// and the last n_tail in s2 chunks of c2. Chunked tiles leave float32 slots
// (dh's first) that head_grad_finish adds in chunk order.
struct GradPlan {
  int n_dh, n_de, n_tail;
  int s1, c1, s2, c2;
  int dh_slots;  // workgroups per dh chunk: n_dh rounded up to a multiple of 8
  int de_slots;  // workgroups of the whole dE tiles, rounded up alike
  int64_t slots() const {
    return (s1 > 1 ? (int64_t)s1 * n_dh : 0) + (s2 > 1 ? (int64_t)s2 * n_tail : 0);
  }
};

// The backward's two products of a token chunk in one launch (the long-K dh
// tiles first): dh[t][c] = sum_v dz[t][v] E[v][c], then
// dE[v][c] (+)= sum_t dz[t][v] h[t][c].
template <bool ACCUM, bool DMA>
__global__ __launch_bounds__(kThreads) void head_grad_kernel(GemmJob dh, GemmJob de, GradPlan pl,
                                                             float* slots) {
  GEMM_LDS_STAGES;
  int b = blockIdx.x;
  const int ndh = pl.s1 * pl.dh_slots;
  if (b < ndh) {
    const int chunk = b / pl.dh_slots, t = b % pl.dh_slots;
    if (t >= pl.n_dh) return;
    const int tile = xcd_tile(t, pl.n_dh, dh.tiles_n);
    const int stages = (dh.A.K + BK - 1) / BK;
    float* slot = pl.s1 > 1 ? slots + ((int64_t)chunk * pl.n_dh + tile) * kSlotElems : nullptr;
    gemm_job<true, false, bf16, false, DMA>(dh, tile, chunk * pl.c1,
                                            min(stages, (chunk + 1) * pl.c1), slot, s0, ring,
                                            threadIdx.x);
    return;
  }
  b -= ndh;
  const int stages = (de.A.K + BK - 1) / BK, n_whole = pl.n_de - pl.n_tail;
  int tile = 0, st0 = 0, st1 = stages;
  float* slot = nullptr;
  if (b < pl.de_slots) {
    if (b >= n_whole) return;
    tile = xcd_tile(b, n_whole, de.tiles_n);
  } else {
    b -= pl.de_slots;
    const int chunk = b / pl.n_tail, t = b % pl.n_tail;
    tile = n_whole + t;
    if (pl.s2 > 1) {
      st0 = chunk * pl.c2;
      st1 = min(stages, st0 + pl.c2);
      slot = slots + ((pl.s1 > 1 ? (int64_t)pl.s1 * pl.n_dh : 0) + (int64_t)chunk * pl.n_tail + t) *
                         kSlotElems;
    }
  }
  gemm_job<false, false, float, ACCUM, DMA>(de, tile, st0, st1, slot, s0, ring, threadIdx.x);
}

// Chunked tiles from their slots, added in chunk order. Block (tile, i * TJ + j)
// takes one 32 x 32 block per wave; dh's tiles come first.
template <bool ACCUM>
__global__ __launch_bounds__(kThreads) void head_grad_finish(GemmJob dh, GemmJob de, GradPlan pl,
                                                             const float* __restrict__ slots) {
  const int n_first = pl.s1 > 1 ? pl.n_dh : 0;
  const int tid = threadIdx.x, ij = blockIdx.y, i = ij / TJ, j = ij % TJ;
  const bool is_dh = (int)blockIdx.x < n_first;
  const int t = is_dh ? blockIdx.x : blockIdx.x - n_first;
  const int n = is_dh ? pl.n_dh : pl.n_tail, s = is_dh ? pl.s1 : pl.s2;
  const float* p = slots + ((is_dh ? 0 : (int64_t)pl.s1 * n_first) + t) * kSlotElems;
  f32x4 v[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = *reinterpret_cast<const f32x4*>(p + slot_at(i, j, q, tid));
  for (int c = 1; c < s; ++c)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const f32x4 u =
          *reinterpret_cast<const f32x4*>(p + (int64_t)c * n * kSlotElems + slot_at(i, j, q, tid));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[q][e] += u[e];
    }
  auto val = [&](int r) { return v[r >> 2][r & 3]; };
  const int tile = is_dh ? t : pl.n_de - pl.n_tail + t;
  if (is_dh)
    put_tile<bf16, false>(dh, tile / dh.tiles_n * BM, tile % dh.tiles_n * BN, i, j, tid, val);
  else
    put_tile<float, ACCUM>(de, tile / de.tiles_n * BM, tile % de.tiles_n * BN, i, j, tid, val);
}

int64_t vpad_of(int V) { return ((int64_t)V + BM - 1) / BM * BM; }

// Token chunk of the backward: bounds the bf16 dz scratch to 2 GiB (all
// 16384 tokens of a 50304-word vocabulary in one chunk), or to
// ALGX_HEAD_CHUNK_BYTES when that is set.
int chunk_tokens(int N, int V) {
  const int64_t per_tok = vpad_of(V) * 2;
  int64_t limit = (int64_t)2 << 30;
  if (const char* env = std::getenv("ALGX_HEAD_CHUNK_BYTES")) {
    const long long v = std::atoll(env);
    if (v > 0) limit = v;
  }
  int64_t c = limit / per_tok;
  c = c / BN * BN;
  if (c < BN) c = BN;
  return (int)(c > N ? ((N + BN - 1) / BN) * BN : c);
}

// Deals the dh and dE tiles of a chunk of ntok tokens. `share` is one compute
// unit's equal part of all k stages. A dh tile runs V / 32 stages, so few
// tokens leave most of the chip idle behind a handful of long tiles: they are
// cut into chunks of about a share. 16 stages or more are aimed at (below that
// the 256 KB a chunk leaves in memory costs more than its products); evened
// out, the chunks of a loop little longer than that have fewer: 17 stages are
// cut in 9 and 8, 33 in 11. At N = 1024, d = 384, V = 32768 (8 dh tiles of 1024 stages) the launch took
// 600 us whole and 72 us in 16 chunks, plus 9 us for adding the slots. With
// many tokens the last dE tiles would run as a partly filled round of whole
// tiles: the ones that no longer fit into a share are cut in chunks of at
// least 128 stages (a chunk's slot, written and read again, costs about 25
// stages): 3088 us whole, 2778 + 7 us so at N = 16384, V = 50304, d = 1024, and
// 2185 whole, 2097 + 35 so at d = 768.
GradPlan grad_plan(int ntok, int d, int V, bool dma) {
  constexpr int kUnits = 256;
  GradPlan pl{};
  const int tn = (d + BN - 1) / BN;
  const int k1 = (V + BK - 1) / BK, k2 = (ntok + BK - 1) / BK;
  pl.n_dh = (ntok + BM - 1) / BM * tn;
  pl.n_de = (V + BM - 1) / BM * tn;
  pl.s1 = pl.s2 = 1;
  pl.c1 = k1;
  pl.c2 = k2;
  if (dma) {
    const int64_t total = (int64_t)pl.n_dh * k1 + (int64_t)pl.n_de * k2;
    const int share = (int)((total + kUnits - 1) / kUnits);
    const int want = share > 16 ? share : 16;
    if (k1 > want) {
      pl.c1 = want;
      pl.s1 = (k1 + want - 1) / want;
      pl.c1 = (k1 + pl.s1 - 1) / pl.s1;
      pl.s1 = (k1 + pl.c1 - 1) / pl.c1;
    }
    // Whole dE tiles that fit beside the dh units within a share.
    const int64_t units = (int64_t)pl.s1 * pl.n_dh;
    const int64_t rounds = units / kUnits, more = units % kUnits;
    auto fit = [&](int64_t busy) { return busy >= share ? 0 : (share - busy) / k2; };
    const int64_t room =
        more * fit((rounds + 1) * pl.c1) + (kUnits - more) * fit(rounds * pl.c1);
    if (k2 >= 256 && room < pl.n_de && room >= kUnits) {
      pl.n_tail = pl.n_de - (int)(room / tn * tn);
      pl.s2 = k2 / 128 < 4 ? k2 / 128 : 4;
      pl.c2 = (k2 + pl.s2 - 1) / pl.s2;
    }
  }
  pl.dh_slots = (pl.n_dh + 7) / 8 * 8;
  pl.de_slots = (pl.n_de - pl.n_tail + 7) / 8 * 8;
  return pl;
}

// dz of a chunk in 32-column blocks ([v / 32][t][32]), read direct-to-LDS by
// the dh/dE launch: dh's 32-wide k stage reads one 64-byte piece per token
// row, dE's reads 32 token rows of one block contiguously (2 KB), instead of
// half lines of 100 KB rows. Needs the operands within the loads' 32-bit
// offsets; else dz is row-major and the launch register-staged.
bool grad_dma(int ntok, int d, int V) {
  const int64_t blk = (int64_t)32 * ntok;
  return dma_span_ok(Operand{nullptr, 32, ntok, V, blk}, true) &&
         dma_span_ok(Operand{nullptr, 32, V, ntok, blk}, false) &&
         dma_span_ok(Operand{nullptr, d, d, V}, false) &&
         dma_span_ok(Operand{nullptr, d, d, ntok}, false);
}

int64_t grad_slot_bytes(int ntok, int d, int V) {
  return grad_plan(ntok, d, V, grad_dma(ntok, d, V)).slots() * kSlotElems * (int64_t)sizeof(float);
}

int32_t check_head(const void* h, const void* E, const int32_t* targets, int N, int d, int V,
                   int kind, int n, int dtype) {
  if (N < 0 || d <= 0 || V <= 0) return fail("head: invalid sizes");
  if (dtype != ALGX_BF16 && dtype != ALGX_F32) return fail("head: dtype must be bf16 or f32");
  if (dtype == ALGX_BF16 && d % 8) return fail("head: hidden width must be a multiple of 8");
  if (kind != ALGX_HEAD_CE && kind != ALGX_HEAD_ALG_CE) return fail("head: unknown kind");
  if (kind == ALGX_HEAD_ALG_CE && (n < 1 || (n & (n - 1)))) return fail("head: n must be a power of two");
  if (N > 0 && (h == nullptr || E == nullptr || targets == nullptr)) return fail("head: null input");
  return 0;
}

typedef void (*HeadFwdFn)(const bf16*, const bf16*, const int32_t*, float*, float*, int, int,
                          int, int, float, float, int);
typedef void (*HeadDzFn)(const bf16*, const bf16*, const int32_t*, const float*, const float*,
                         bf16*, int64_t, int64_t, int, int, int, int, int, float, float, int);

// Kernel instance for (kind, n): alg_ce with n = 8, 16 or 32 gets unrolled
// powers in both kernels, and the forward also for n = 2, 4 and 64 (its
// runtime power loop, kept for n >= 128, spills registers). DMA (the
// direct-to-LDS ring) when d is a multiple of BK.
template <bool DMA> HeadFwdFn pick_head_fwd_as(int kind, int log2n) {
  if (kind == ALGX_HEAD_CE) return head_fwd_kernel<ALGX_HEAD_CE, 0, DMA>;
  switch (log2n) {
    case 1: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 1, DMA>;
    case 2: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 2, DMA>;
    case 3: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 3, DMA>;
    case 4: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 4, DMA>;
    case 5: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 5, DMA>;
    case 6: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 6, DMA>;
    default: return head_fwd_kernel<ALGX_HEAD_ALG_CE, 0, DMA>;
  }
}
template <bool DMA, bool BLK> HeadDzFn pick_head_dz_as(int kind, int log2n) {
  if (kind == ALGX_HEAD_CE) return head_dz_kernel<ALGX_HEAD_CE, 0, DMA, BLK>;
  switch (log2n) {
    case 3: return head_dz_kernel<ALGX_HEAD_ALG_CE, 3, DMA, BLK>;
    case 4: return head_dz_kernel<ALGX_HEAD_ALG_CE, 4, DMA, BLK>;
    case 5: return head_dz_kernel<ALGX_HEAD_ALG_CE, 5, DMA, BLK>;
    default: return head_dz_kernel<ALGX_HEAD_ALG_CE, 0, DMA, BLK>;
  }
}
// The logit products run direct-to-LDS when d is a whole number of ring
// turns and E and the token rows fit the loads' 32-bit offsets.
bool logits_dma(int d, int V, int ntok) {
  return d % (BK * kDmaStages) == 0 && dma_span_ok(Operand{nullptr, d, V, d}, true) &&
         dma_span_ok(Operand{nullptr, d, ntok, d}, true);
}
HeadFwdFn pick_head_fwd(int kind, int log2n, int d, int V, int N) {
  return logits_dma(d, V, N) ? pick_head_fwd_as<true>(kind, log2n)
                             : pick_head_fwd_as<false>(kind, log2n);
}
HeadDzFn pick_head_dz(int kind, int log2n, int d, bool blocked, int V, int ntok) {
  const bool dma = logits_dma(d, V, ntok);
  if (blocked)
    return dma ? pick_head_dz_as<true, true>(kind, log2n) : pick_head_dz_as<false, true>(kind, log2n);
  return dma ? pick_head_dz_as<true, false>(kind, log2n) : pick_head_dz_as<false, false>(kind, log2n);
}

// Vocabulary tiles per forward workgroup: the token blocks x vocabulary tiles
// dealt out in about kFwdWorkgroups equal chunks (one round of the CUs), so
// no partial last round of workgroups is left.
int chunk_tiles_of(int N, int V) {
  const int64_t ntv = (V + BM - 1) / BM, ntb = (N + BN - 1) / BN;
  const int64_t per = (ntv * ntb + kFwdWorkgroups - 1) / kFwdWorkgroups;
  const int64_t nch = (ntv + per - 1) / per;
  return (int)((ntv + nch - 1) / nch);
}
int nchunks_of(int N, int V) {
  const int nt = (V + BM - 1) / BM, ct = chunk_tiles_of(N, V);
  return (nt + ct - 1) / ct;
}

}  // namespace
}  // namespace algx

using namespace algx;

namespace {

int64_t fwd_partial_bytes(int32_t N, int32_t V, int32_t dtype) {
  if (N <= 0 || V <= 0) return 0;
  if (dtype == ALGX_F32) return head_f32_fwd_workspace(N, V);
  return (int64_t)nchunks_of(N, V) * N * 2 * sizeof(float);
}

int stat_blocks(int N) { return (N + kStatTokens - 1) / kStatTokens; }

// The forward up to stat and zt, and with tel the telemetry and objective
// (obj_part: stat_blocks(N) floats).
int32_t head_forward(const void* h, const void* E, const int32_t* targets, float* stat, float* zt,
                     float* tel, float* obj, float* partial, float* obj_part, int32_t N, int32_t d,
                     int32_t V, int32_t kind, int32_t n, float inv_c, float clamp, int32_t dtype,
                     hipStream_t s) {
  const int log2n = kind == ALGX_HEAD_ALG_CE ? ilog2(n) : 0;
  int nch;
  if (dtype == ALGX_F32) {
    if (int32_t rc = head_f32_fwd((const float*)h, (const float*)E, targets, zt, partial, N, d, V,
                                  kind, log2n, inv_c, clamp, &nch, s))
      return rc;
  } else {
    nch = nchunks_of(N, V);
    dim3 grid((N + BN - 1) / BN, nch);
    launch_k(probe_for(ALGX_PROBE_HEAD_FWD), pick_head_fwd(kind, log2n, d, V, N), grid,
             dim3(kThreads), s, (const bf16*)h, (const bf16*)E, targets, zt, partial, N, d, V,
             log2n, inv_c, clamp, chunk_tiles_of(N, V));
    if (int32_t rc = check_launch("head_fwd")) return rc;
  }
  const HeadStat p{partial, targets, zt, stat, tel, obj_part, nch, N, V, log2n, inv_c, clamp};
  const int nb = stat_blocks(N);
  if (kind == ALGX_HEAD_CE)
    head_stat_kernel<ALGX_HEAD_CE><<<nb, 256, 0, s>>>(p);
  else
    head_stat_kernel<ALGX_HEAD_ALG_CE><<<nb, 256, 0, s>>>(p);
  if (int32_t rc = check_launch("head_stat")) return rc;
  if (tel == nullptr) return 0;
  head_mean_kernel<<<1, 256, 0, s>>>(obj_part, nb, N, obj);
  return check_launch("head_mean");
}

}  // namespace

extern "C" int64_t algx_head_fwd_workspace_bytes(int32_t N, int32_t d, int32_t V, int32_t dtype) {
  (void)d;
  return fwd_partial_bytes(N, V, dtype);
}

extern "C" int32_t algx_head_fwd(const void* h, const void* E, const int32_t* targets,
                                 float* stat, float* zt, void* workspace, int32_t N, int32_t d,
                                 int32_t V, int32_t kind, int32_t n, float inv_c, float clamp,
                                 int32_t dtype, void* stream) {
  if (int32_t rc = check_head(h, E, targets, N, d, V, kind, n, dtype)) return rc;
  if (N == 0) return 0;
  if (stat == nullptr || zt == nullptr || workspace == nullptr) return fail("head_fwd: null output");
  return head_forward(h, E, targets, stat, zt, nullptr, nullptr, (float*)workspace, nullptr, N, d,
                      V, kind, n, inv_c, clamp, dtype, (hipStream_t)stream);
}

extern "C" int64_t algx_head_loss_workspace_bytes(int32_t N, int32_t d, int32_t V, int32_t dtype) {
  (void)d;
  if (N <= 0 || V <= 0) return 0;
  // the chunk partials, the target logits, the objective's shares
  return fwd_partial_bytes(N, V, dtype) + ((int64_t)N + stat_blocks(N)) * (int64_t)sizeof(float);
}

extern "C" int32_t algx_head_loss(const void* h, const void* E, const int32_t* targets,
                                  float* stat, float* tel, float* obj, void* workspace, int32_t N,
                                  int32_t d, int32_t V, int32_t kind, int32_t n, float inv_c,
                                  float clamp, int32_t dtype, void* stream) {
  if (int32_t rc = check_head(h, E, targets, N, d, V, kind, n, dtype)) return rc;
  if (N == 0) return fail("head_loss: the mean over no tokens");
  if (stat == nullptr || tel == nullptr || obj == nullptr || workspace == nullptr)
    return fail("head_loss: null output");
  float* partial = (float*)workspace;
  float* zt = (float*)((char*)workspace + fwd_partial_bytes(N, V, dtype));
  return head_forward(h, E, targets, stat, zt, tel, obj, partial, zt + N, N, d, V, kind, n, inv_c,
                      clamp, dtype, (hipStream_t)stream);
}

extern "C" int64_t algx_head_bwd_workspace_bytes(int32_t N, int32_t d, int32_t V, int32_t dtype) {
  if (N <= 0 || V <= 0) return 0;
  if (dtype == ALGX_F32) return head_f32_bwd_workspace(N, d > 0 ? d : 0, V);
  const int csize = chunk_tokens(N, V);
  const int64_t dz = (int64_t)csize * vpad_of(V) * 2;
  if (d <= 0) return dz;
  // the slots of the full token chunks and of the last one
  const int first = csize < N ? csize : N, last = N - (N - 1) / csize * csize;
  const int64_t sf = grad_slot_bytes(first, d, V), sl = grad_slot_bytes(last, d, V);
  return dz + (sf > sl ? sf : sl);
}

extern "C" int32_t algx_head_bwd(const void* h, const void* E, const int32_t* targets,
                                 const float* stat, const float* scale, void* dh, float* dE,
                                 void* workspace, int32_t N, int32_t d, int32_t V, int32_t kind,
                                 int32_t n, float inv_c, float clamp, int32_t dtype,
                                 void* stream) {
  if (int32_t rc = check_head(h, E, targets, N, d, V, kind, n, dtype)) return rc;
  hipStream_t s = (hipStream_t)stream;
  if (dE == nullptr) return fail("head_bwd: null dE");
  if (N == 0) return fill_f32(dE, (int64_t)V * d, 0.0f, s);
  if (stat == nullptr || scale == nullptr || dh == nullptr || workspace == nullptr)
    return fail("head_bwd: null pointer");
  const int log2n = kind == ALGX_HEAD_ALG_CE ? ilog2(n) : 0;
  if (dtype == ALGX_F32)
    return head_f32_bwd((const float*)h, (const float*)E, targets, stat, scale, (float*)dh, dE,
                        (float*)workspace, N, d, V, kind, log2n, inv_c, clamp, s);
  const int64_t ldz = vpad_of(V);
  const int csize = chunk_tokens(N, V);
  bf16* dz = (bf16*)workspace;
  float* slots = (float*)((char*)workspace + (int64_t)csize * ldz * 2);
  const bf16* hb = (const bf16*)h;
  const bf16* eb = (const bf16*)E;
  for (int tok0 = 0; tok0 < N; tok0 += csize) {
    const int ntok = min(csize, N - tok0);
    const int ct = chunk_tiles_of(ntok, V);
    const int64_t blk = (int64_t)32 * ntok;
    const bool dma = grad_dma(ntok, d, V);
    const int64_t bstride = dma ? blk : 0;
    dim3 gdz((ntok + BN - 1) / BN, ((V + BM - 1) / BM + ct - 1) / ct);
    launch_k(probe_for(ALGX_PROBE_HEAD_DZ),
             pick_head_dz(kind, log2n, d, bstride != 0, V, ntok),
             gdz, dim3(kThreads), s, hb, eb, targets, stat, scale, dz, ldz, bstride, tok0, ntok, d,
             V, log2n, inv_c, clamp, ct);
    if (int32_t rc = check_launch("head_dz")) return rc;
    // dh[t][c] = sum_v dz[t][v] E[v][c]: A = dz (k-contiguous), B(n=c,k=v) = E stored [v][c].
    // dE[v][c] (+)= sum_t dz[t][v] h[t][c]: A(m=v,k=t) = dz stored [t][v], B(n=c,k=t) = h [t][c].
    const int tn = (d + BN - 1) / BN;
    const Operand dz_t = dma ? Operand{dz, 32, ntok, V, bstride} : Operand{dz, ldz, ntok, V};
    const Operand dz_v = dma ? Operand{dz, 32, V, ntok, bstride} : Operand{dz, ldz, V, ntok};
    const GemmJob jdh{dz_t, Operand{eb, d, d, V}, (bf16*)dh + (int64_t)tok0 * d, (int64_t)d,
                      ntok, d, tn};
    const GemmJob jde{dz_v, Operand{hb + (int64_t)tok0 * d, d, d, ntok}, dE, (int64_t)d, V, d, tn};
    const GradPlan pl = grad_plan(ntok, d, V, dma);
    auto gk = dma ? (tok0 == 0 ? head_grad_kernel<false, true> : head_grad_kernel<true, true>)
                  : (tok0 == 0 ? head_grad_kernel<false, false> : head_grad_kernel<true, false>);
    const int grid = pl.s1 * pl.dh_slots + pl.de_slots + pl.s2 * pl.n_tail;
    launch_k(probe_for(ALGX_PROBE_HEAD_DE), gk, dim3(grid), dim3(kThreads), s, jdh, jde, pl, slots);
    if (int32_t rc = check_launch("head_grad")) return rc;
    const int nsplit = (pl.s1 > 1 ? pl.n_dh : 0) + (pl.s2 > 1 ? pl.n_tail : 0);
    if (nsplit > 0) {
      auto fk = tok0 == 0 ? head_grad_finish<false> : head_grad_finish<true>;
      launch_k(Probe{}, fk, dim3(nsplit, TI * TJ), dim3(kThreads), s, jdh, jde, pl,
               (const float*)slots);
      if (int32_t rc = check_launch("head_grad_finish")) return rc;
    }
  }
  return 0;
}
