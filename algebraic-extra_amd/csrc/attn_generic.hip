// Generic attention kernels: every numeric variant of flash.py, float32 or
// bf16 storage, D in {16, 32, 64}, any T. They carry the float32 path and the
// head widths the bf16 MFMA kernels do not take. Numerics follow
// flash.py:189-284 (forward) and flash.py:333-361 (tile VJP), with the
// reference's rounding points: p -> storage dtype before PV and dV, ds ->
// storage dtype before dK and dQ, outputs cast at the end; every product and
// sum is float32.
//
// A workgroup of 4 waves owns 16 rows of one head (queries in the forward and
// dQ, keys in dK/dV) and its waves share out the 16-row tiles of the other
// side, each with accumulators (and running maximum) of its own that are
// merged through LDS at the end. The products run on
// v_mfma_f32_16x16x4_f32: lane l = 16 g + c holds A[c][g], B[g][c] and, in
// accumulator register i, C[4 g + i][c]. Which of a contraction's indices sits
// in which k-slot is free as long as both operands agree, so no operand passes
// through LDS:
//   scores   slot (step s, g) is d = D/4 g + s: a lane reads D/4 consecutive
//            values of row c of each side.
//   updates  slot (step i, g) is tile row 4 g + i, the rows whose weights the
//            lane holds: the weights are the B operand as they stand, and the
//            A operand's row m stands for d = D/16 m + dt, so a lane reads D/16
//            consecutive values of rows 4 g + i. Its D/4 accumulators are then
//            D/4 consecutive values of its column's row, from D/4 g.
// Bound by the matrix units and by the loads in front of them: with one tile
// per wave in flight, a wave loads the next tile's operands before the current
// tile's products. Measured against the one-thread-per-row kernels these
// replace (whose chains of D FMAs per score left all but a few CUs idle),
// float32 guarded calls: B=1, H=4, T=256 forward, a whole call, 285 -> 18 us (its
// three kernels 15.4, this one 9.4); B=2, H=12, T=512, these kernels alone,
// forward 575 -> 27 us, dK/dV and dQ 1223 -> 94 us. A guarded call is one launch
// of each, which chooses the variant: with one launch per variant the first
// call took 21 us. The distance from float64 did not grow (5.9e-7 ->
// 5.6e-7 of o at the first shape).
#include "attn_aux.h"

namespace algx {

namespace {

constexpr int kRows = 16;   // rows per workgroup and per tile
constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// N consecutive elements as float32.
template <typename T, int N>
__device__ __forceinline__ void load_run(const T* p, float (&out)[N]) {
  constexpr int bytes = N * (int)sizeof(T), V = bytes < 16 ? N : 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(V)));
#pragma unroll
  for (int i = 0; i < N / V; ++i) {
    if constexpr (V == 1) {
      out[i] = to_f(p[i]);
    } else {
      const vec x = *reinterpret_cast<const vec*>(p + i * V);
#pragma unroll
      for (int e = 0; e < V; ++e) out[i * V + e] = to_f(x[e]);
    }
  }
}

// Score operand of a tile: row row0 + c, values D/4 g .. (zero past T_).
template <typename T, int D>
__device__ __forceinline__ void load_rows(const T* head, int row0, int T_, int c, int g,
                                          float (&out)[D / 4]) {
  const int row = row0 + c;
  load_run(head + (int64_t)min(row, T_ - 1) * D + D / 4 * g, out);
  if (row >= T_)
#pragma unroll
    for (int i = 0; i < D / 4; ++i) out[i] = 0.0f;
}

// Update operand of a tile: rows row0 + 4 g + i, values D/16 c .. (zero past T_).
template <typename T, int D>
__device__ __forceinline__ void load_cols(const T* head, int row0, int T_, int c, int g,
                                          float (&out)[4][D / 16]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = row0 + 4 * g + i;
    load_run(head + (int64_t)min(row, T_ - 1) * D + D / 16 * c, out[i]);
    if (row >= T_)
#pragma unroll
      for (int e = 0; e < D / 16; ++e) out[i][e] = 0.0f;
  }
}

// Products of 16 rows of each side: C[4 g + i][c] = sum_d a(4 g + i) b(c).
template <int N>
__device__ __forceinline__ f32x4 scores(const float (&a)[N], const float (&b)[N]) {
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int s = 0; s < N; ++s) acc = mfma4(a[s], b[s], acc);
  return acc;
}

// acc += sum over the tile's rows of w(row, c) x(row).
template <int D>
__device__ __forceinline__ void update(const float (&x)[4][D / 16], const float (&w)[4],
                                       f32x4 (&acc)[D / 16]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int dt = 0; dt < D / 16; ++dt) acc[dt] = mfma4(x[i][dt], w[i], acc[dt]);
}

// update() of a tile on the diagonal, where row row0 + j counts for column c
// only if seen(j). A masked row's weight is 0, but 0 times an infinity or NaN
// of that row would not be: a tile that holds one is summed row by row over
// the visible ones.
template <typename T, int D, typename Seen>
__device__ __forceinline__ void update_diag(const T* head, int row0, int T_, int c, int g,
                                            const float (&x)[4][D / 16], const float (&w)[4],
                                            f32x4 (&acc)[D / 16], Seen&& seen) {
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int e = 0; e < D / 16; ++e)
      bad |= !(__builtin_fabsf(x[i][e]) < __builtin_inff());
  if (!__any(bad)) {
    update<D>(x, w, acc);
    return;
  }
#pragma unroll 1
  for (int j = 0; j < kRows; ++j) {
    if (row0 + j >= T_) break;
    const int r = j & 3;
    const float mine = r == 0 ? w[0] : r == 1 ? w[1] : r == 2 ? w[2] : w[3];
    const float wj = __shfl(mine, (j >> 2) * 16 + c, 64);
    float row[D / 4];
    load_run(head + (int64_t)(row0 + j) * D + D / 4 * g, row);
    if (seen(j))
#pragma unroll
      for (int e = 0; e < D / 4; ++e)
        acc[e % (D / 16)][e / (D / 16)] =
            __builtin_fmaf(wj, row[e], acc[e % (D / 16)][e / (D / 16)]);
  }
}

// A wave's accumulators (D/4 values of column c's row, from D/4 g) to LDS.
template <int D>
__device__ __forceinline__ void put_acc(float (*dst)[D + 4], const f32x4 (&acc)[D / 16], int c,
                                        int g) {
#pragma unroll
  for (int e = 0; e < D / 4; ++e) dst[c][D / 4 * g + e] = acc[e % (D / 16)][e / (D / 16)];
}

__device__ __forceinline__ float over_groups_max(float v) {
  v = __builtin_fmaxf(v, __shfl_xor(v, 16, 64));
  return __builtin_fmaxf(v, __shfl_xor(v, 32, 64));
}

// exp(m - to) or (rho(m) rho(-to))^n: the factor that moves sums taken at
// maximum m to the maximum `to`; nothing summed yet (m = -inf): 0.
__device__ __forceinline__ float rescale(const KVariant& var, float m, float to) {
  if (m == -__builtin_inff()) return 0.0f;
  if (var.kind == ALGX_SOFTMAX) return __expf(m - to);
  float r;
  return pow2n(rho_exact(m, r) * rho_exact(-to, r), var.log2n);
}

template <typename T, int D>
__global__ __launch_bounds__(kThreads) void fwd_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const float* __restrict__ sink, T* __restrict__ o, float* __restrict__ o_precise,
    float* __restrict__ stat, int H, int T_, KVariant lo, KVariant hi,
    const int32_t* __restrict__ guard) {
  const KVariant var = guard_in_range(guard) ? lo : hi;
  __shared__ float acc_s[kWaves][kRows][D + 4];
  __shared__ float m_s[kWaves][kRows], l_s[kWaves][kRows];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int bh = blockIdx.y, h = bh % H;
  const int qb = gridDim.x - 1 - blockIdx.x;  // most keys first
  const int64_t base = (int64_t)bh * T_ * D;
  const T* kh = k + base;
  const T* vh = v + base;
  float qf[D / 4];
  load_rows<T, D>(q + base, qb * kRows, T_, c, g, qf);
  const bool noshift = var.kind == ALGX_ASINH && !var.shift;
  // The sink is one more term of the row, carried by wave 0 (lanes g = 0).
  float m = noshift ? 0.0f : -__builtin_inff(), l = 0.0f;
  if (w == 0 && sink != nullptr) {
    float l0;
    sink_init(var, true, var.sink(sink, h), m, l0);
    l = g == 0 ? l0 : 0.0f;
  }
  f32x4 acc[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) acc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  float kf[D / 4], vf[4][D / 16];
  auto load = [&](int kt) {
    load_rows<T, D>(kh, kt * kRows, T_, c, g, kf);
    load_cols<T, D>(vh, kt * kRows, T_, c, g, vf);
  };
  if (w <= qb) load(w);
  for (int kt = w; kt <= qb; kt += kWaves) {
    float kc[D / 4], vc[4][D / 16];
#pragma unroll
    for (int e = 0; e < D / 4; ++e) {
      kc[e] = kf[e];
      vc[e / (D / 16)][e % (D / 16)] = vf[e / (D / 16)][e % (D / 16)];
    }
    if (kt + kWaves <= qb) load(kt + kWaves);
    const f32x4 s = scores(kc, qf);
    const bool diag = kt == qb;
    float p[4];
    float lsum = 0.0f;
    if (noshift) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = var.bounded ? s[i] : __builtin_fminf(s[i], var.clamp);
        float r;
        p[i] = pow2n(rho_of(var, x, r), var.log2n);
        if (diag && 4 * g + i > c) p[i] = 0.0f;
        lsum += p[i];
      }
      l += lsum;
    } else {
      float tmax = -__builtin_inff();
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(diag && 4 * g + i > c)) tmax = __builtin_fmaxf(tmax, s[i]);
      const float m_new = __builtin_fmaxf(m, over_groups_max(tmax));
      const float alpha = rescale(var, m, m_new);
      float r, shf = 0.0f;
      if (var.kind != ALGX_SOFTMAX) shf = rho_exact(-m_new, r);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = var.kind == ALGX_SOFTMAX ? __expf(s[i] - m_new)
                                        : pow2n(rho_var(s[i], var.fast, r) * shf, var.log2n);
        // A score of -inf weighs nothing, also where the wave has met no other
        // score yet (m_new = -inf): a row is NaN only if all its scores are.
        if ((diag && 4 * g + i > c) || s[i] == -__builtin_inff()) p[i] = 0.0f;
        lsum += p[i];
      }
      l = l * alpha + lsum;
#pragma unroll
      for (int dt = 0; dt < D / 16; ++dt)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) acc[dt][r4] *= alpha;
      m = m_new;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = round_to<T>(p[i]);
    if (diag)
      update_diag<T, D>(vh, kt * kRows, T_, c, g, vc, p, acc, [&](int j) { return j <= c; });
    else
      update<D>(vc, p, acc);
  }

  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) {
    m_s[w][c] = m;
    l_s[w][c] = l;
  }
  put_acc<D>(acc_s[w], acc, c, g);
  __syncthreads();
  // Thread -> 4 consecutive values of one row.
  if (tid >= kRows * D / 4) return;
  const int r = tid / (D / 4), d0 = 4 * (tid % (D / 4));
  const int i = qb * kRows + r;
  if (i >= T_) return;
  float mt = m_s[0][r];
#pragma unroll
  for (int ww = 1; ww < kWaves; ++ww) mt = __builtin_fmaxf(mt, m_s[ww][r]);
  float lt = 0.0f;
  f32x4 val = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int ww = 0; ww < kWaves; ++ww) {
    const float f = noshift ? 1.0f : rescale(var, m_s[ww][r], mt);
    lt = __builtin_fmaf(l_s[ww][r], f, lt);
#pragma unroll
    for (int e = 0; e < 4; ++e) val[e] = __builtin_fmaf(acc_s[ww][r][d0 + e], f, val[e]);
  }
  const float inv = 1.0f / lt;
  const int64_t at = base + (int64_t)i * D + d0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[at + e] = from_f<T>(val[e] * inv);
    if (var.precise && o_precise != nullptr) o_precise[at + e] = val[e] * inv;
  }
  if (d0 == 0) stat[(int64_t)bh * T_ + i] = final_stat(var, mt, lt);
}

// dK, dV of 16 keys: query tiles from the keys' own onwards.
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void bwd_dkdv_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const float* __restrict__ stat, const float* __restrict__ di, const T* __restrict__ dout,
    T* __restrict__ dk, T* __restrict__ dv, int T_, KVariant lo,
    KVariant hi, const int32_t* __restrict__ guard) {
  const KVariant var = guard_in_range(guard) ? lo : hi;
  __shared__ float dk_s[kWaves][kRows][D + 4], dv_s[kWaves][kRows][D + 4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int bh = blockIdx.y, kb = blockIdx.x;  // most queries first
  const int64_t base = (int64_t)bh * T_ * D, rbase = (int64_t)bh * T_;
  const T* qh = q + base;
  const T* gh = dout + base;
  float kf[D / 4], vf[D / 4];
  load_rows<T, D>(k + base, kb * kRows, T_, c, g, kf);
  load_rows<T, D>(v + base, kb * kRows, T_, c, g, vf);
  f32x4 dka[D / 16], dva[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) dka[dt] = dva[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool asinh = var.kind == ALGX_ASINH;
  const int nqt = (T_ + kRows - 1) / kRows;
  for (int qt = kb + w; qt < nqt; qt += kWaves) {
    const int q0 = qt * kRows;
    float qr[D / 4], gr[D / 4], qc[4][D / 16], gc[4][D / 16];
    load_rows<T, D>(qh, q0, T_, c, g, qr);
    load_rows<T, D>(gh, q0, T_, c, g, gr);
    load_cols<T, D>(qh, q0, T_, c, g, qc);
    load_cols<T, D>(gh, q0, T_, c, g, gc);
    float st[4], dd[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int at = min(q0 + 4 * g + i, T_ - 1);
      st[i] = stat[rbase + at];
      dd[i] = di[rbase + at];
    }
    const f32x4 s = scores(qr, kf), dp = scores(gr, vf);
    const bool diag = qt == kb;
    float p[4], ds[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float rr;
      bool keep;
      p[i] = bwd_weight(var, s[i], st[i], rr, keep);
      ds[i] = p[i] * (dp[i] - dd[i]);
      if (asinh) ds[i] = keep ? ds[i] * rr : 0.0f;
      if (q0 + 4 * g + i >= T_ || (diag && 4 * g + i < c)) p[i] = ds[i] = 0.0f;
      p[i] = round_to<T>(p[i]);
      ds[i] = round_to<T>(ds[i]);
    }
    if (diag) {
      auto seen = [&](int j) { return j >= c; };
      update_diag<T, D>(gh, q0, T_, c, g, gc, p, dva, seen);
      update_diag<T, D>(qh, q0, T_, c, g, qc, ds, dka, seen);
    } else {
      update<D>(gc, p, dva);
      update<D>(qc, ds, dka);
    }
  }
  put_acc<D>(dk_s[w], dka, c, g);
  put_acc<D>(dv_s[w], dva, c, g);
  __syncthreads();
  if (tid >= kRows * D / 4) return;
  const int r = tid / (D / 4), d0 = 4 * (tid % (D / 4));
  const int j = kb * kRows + r;
  if (j >= T_) return;
  const int64_t at = base + (int64_t)j * D + d0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float sk = (dk_s[0][r][d0 + e] + dk_s[1][r][d0 + e]) +
                     (dk_s[2][r][d0 + e] + dk_s[3][r][d0 + e]);
    const float sv = (dv_s[0][r][d0 + e] + dv_s[1][r][d0 + e]) +
                     (dv_s[2][r][d0 + e] + dv_s[3][r][d0 + e]);
    dk[at + e] = from_f<T>(sk * var.slope);
    dv[at + e] = from_f<T>(sv);
  }
}

// dQ of 16 queries: key tiles up to the diagonal. Writes the final
// dq = cast(cast(dq_s * slope) * q_scale).
template <typename T, int D>
__global__ __launch_bounds__(kThreads) void bwd_dq_generic_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v,
    const float* __restrict__ stat, const float* __restrict__ di, const T* __restrict__ dout,
    T* __restrict__ dq, int T_, float q_scale, KVariant lo, KVariant hi,
    const int32_t* __restrict__ guard) {
  const KVariant var = guard_in_range(guard) ? lo : hi;
  __shared__ float dq_s[kWaves][kRows][D + 4];
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int bh = blockIdx.y, qb = gridDim.x - 1 - blockIdx.x;
  const int64_t base = (int64_t)bh * T_ * D;
  const T* kh = k + base;
  const T* vh = v + base;
  float qf[D / 4], gf[D / 4];
  load_rows<T, D>(q + base, qb * kRows, T_, c, g, qf);
  load_rows<T, D>(dout + base, qb * kRows, T_, c, g, gf);
  const int64_t srow = (int64_t)bh * T_ + min(qb * kRows + c, T_ - 1);
  const float st = stat[srow], dd = di[srow];
  f32x4 acc[D / 16];
#pragma unroll
  for (int dt = 0; dt < D / 16; ++dt) acc[dt] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool asinh = var.kind == ALGX_ASINH;
  for (int kt = w; kt <= qb; kt += kWaves) {
    const int k0 = kt * kRows;
    float kr[D / 4], vr[D / 4], kc[4][D / 16];
    load_rows<T, D>(kh, k0, T_, c, g, kr);
    load_rows<T, D>(vh, k0, T_, c, g, vr);
    load_cols<T, D>(kh, k0, T_, c, g, kc);
    const f32x4 s = scores(kr, qf), dp = scores(vr, gf);
    const bool diag = kt == qb;
    float ds[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float rr;
      bool keep;
      const float p = bwd_weight(var, s[i], st, rr, keep);
      ds[i] = p * (dp[i] - dd);
      if (asinh) ds[i] = keep ? ds[i] * rr : 0.0f;
      if (diag && 4 * g + i > c) ds[i] = 0.0f;
      ds[i] = round_to<T>(ds[i]);
    }
    if (diag)
      update_diag<T, D>(kh, k0, T_, c, g, kc, ds, acc, [&](int j) { return j <= c; });
    else
      update<D>(kc, ds, acc);
  }
  put_acc<D>(dq_s[w], acc, c, g);
  __syncthreads();
  if (tid >= kRows * D / 4) return;
  const int r = tid / (D / 4), d0 = 4 * (tid % (D / 4));
  const int i = qb * kRows + r;
  if (i >= T_) return;
  const int64_t at = base + (int64_t)i * D + d0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float sum = (dq_s[0][r][d0 + e] + dq_s[1][r][d0 + e]) +
                      (dq_s[2][r][d0 + e] + dq_s[3][r][d0 + e]);
    dq[at + e] = from_f<T>(round_to<T>(sum * var.slope) * q_scale);
  }
}

}  // namespace

int32_t launch_fwd_generic(const void* q, const void* k, const void* v, const float* sink,
                           void* o, float* o_precise, float* stat, int B, int H, int T, int D,
                           int dtype, const KVariant& lo, const KVariant& hi, const int32_t* guard,
                           hipStream_t s) {
  dim3 grid((T + kRows - 1) / kRows, B * H);
#define FWD_CASE(TT, DD)                                                                         \
  fwd_generic_kernel<TT, DD><<<grid, kThreads, 0, s>>>((const TT*)q, (const TT*)k, (const TT*)v, \
                                                       sink, (TT*)o, o_precise, stat, H, T, lo,  \
                                                       hi, guard)
  if (dtype == ALGX_BF16) {
    if (D == 64) FWD_CASE(bf16, 64);
    else if (D == 32) FWD_CASE(bf16, 32);
    else if (D == 16) FWD_CASE(bf16, 16);
    else return fail("attn_fwd: D must be 16, 32 or 64");
  } else {
    if (D == 64) FWD_CASE(float, 64);
    else if (D == 32) FWD_CASE(float, 32);
    else if (D == 16) FWD_CASE(float, 16);
    else return fail("attn_fwd: D must be 16, 32 or 64");
  }
#undef FWD_CASE
  return check_launch("attn_fwd_generic");
}

int32_t launch_bwd_generic(const void* q, const void* k, const void* v, const float* stat,
                           const float* di, const void* dout, void* dq, void* dk, void* dv,
                           int B, int H, int T, int D, int dtype, float q_scale,
                           const KVariant& lo, const KVariant& hi, const int32_t* guard,
                           hipStream_t s) {
  dim3 grid((T + kRows - 1) / kRows, B * H);
#define BWD_CASE(TT, DD)                                                                        \
  do {                                                                                          \
    bwd_dkdv_generic_kernel<TT, DD><<<grid, kThreads, 0, s>>>(                                  \
        (const TT*)q, (const TT*)k, (const TT*)v, stat, di, (const TT*)dout, (TT*)dk, (TT*)dv, \
        T, lo, hi, guard);                                                                      \
    bwd_dq_generic_kernel<TT, DD><<<grid, kThreads, 0, s>>>((const TT*)q, (const TT*)k,         \
                                                            (const TT*)v, stat, di,             \
                                                            (const TT*)dout, (TT*)dq, T,        \
                                                            q_scale, lo, hi, guard);            \
  } while (0)
  if (dtype == ALGX_BF16) {
    if (D == 64) BWD_CASE(bf16, 64);
    else if (D == 32) BWD_CASE(bf16, 32);
    else if (D == 16) BWD_CASE(bf16, 16);
    else return fail("attn_bwd: D must be 16, 32 or 64");
  } else {
    if (D == 64) BWD_CASE(float, 64);
    else if (D == 32) BWD_CASE(float, 32);
    else if (D == 16) BWD_CASE(float, 16);
    else return fail("attn_bwd: D must be 16, 32 or 64");
  }
#undef BWD_CASE
  return check_launch("attn_bwd_generic");
}

}  // namespace algx
