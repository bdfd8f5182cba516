// The operators' autograd functions over the C ABI (include/algx.h), for
// PyTorch: allocation, argument marshalling and the backward's node in native
// code. The Python modules of the same operators check their arguments and call
// these; the device work is libalgx.so's.
//
// As Python functions over ctypes, a forward and backward cost the host more
// than the kernels of most calls take (the engine's thread taking the
// interpreter lock, some ten allocations and twenty converted arguments each
// way). With the same kernels, forward and backward: qk_rms_norm_pair at
// [8, 2048, 16, 64] 155 -> 77 us, softmax attention at B=8, H=6, T=1024
// 163 -> 80 us, a guarded one at B=2, H=12, T=333 231 -> 108 us.
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <optional>
#include <tuple>

#include "algx.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Function;
using torch::autograd::variable_list;

void* stream() { return c10::hip::getCurrentHIPStream().stream(); }

void check(int32_t rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed (", rc, "): ", algx_last_error());
}

int32_t dtype_code(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return ALGX_BF16;
  TORCH_CHECK_VALUE(t.scalar_type() == at::kFloat, "unsupported dtype ", t.scalar_type());
  return ALGX_F32;
}

void on_device(const Tensor& t, const char* what) {
  TORCH_CHECK(t.is_cuda(), what, " needs tensors on the GPU");
}

void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }

Tensor f32(at::IntArrayRef shape, const Tensor& like) {
  return at::empty(shape, like.options().dtype(at::kFloat));
}
Tensor scratch(int64_t bytes, const Tensor& like) {
  return at::empty({bytes > 0 ? bytes : 1}, like.options().dtype(at::kByte));
}

// Contiguous with a 16-byte aligned base (the kernels move 16-byte vectors).
Tensor aligned(const Tensor& t) {
  Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone();
}
Tensor grad_like(const Tensor& g, const Tensor& x) {
  return g.defined() ? g.to(x.scalar_type()).contiguous() : at::zeros_like(x);
}
Tensor aligned_grad(const Tensor& g, const Tensor& x) {
  return g.defined() ? aligned(g.to(x.scalar_type())) : at::zeros_like(x);
}
Tensor gain32(const std::optional<Tensor>& g) {
  return g.has_value() ? g->to(at::kFloat).contiguous() : Tensor();
}
std::optional<Tensor> opt(const Tensor& t) {
  return t.defined() ? std::optional<Tensor>(t) : std::nullopt;
}
int64_t rows_of(const Tensor& x) {
  const int64_t D = x.size(-1);
  return D > 0 ? x.numel() / D : 0;
}

// ---------------------------------------------------------------- attention

// What flash_attention derives from its options (kernels/flash.py).
struct FlashPlan : torch::CustomClassHolder {
  algx_attn_variant low{}, high{};
  bool guarded = false;
  double scale = 1.0, bound = 0.0, vmax = 0.0;
  const algx_attn_variant* hi() const { return guarded ? &high : nullptr; }
  bool precise() const { return low.precise_output || (guarded && high.precise_output); }
};
using PlanPtr = c10::intrusive_ptr<FlashPlan>;
typedef std::tuple<int, int, int, int, int, int, int, double, int> VariantFields;

algx_attn_variant variant(const VariantFields& f) {
  algx_attn_variant v{};
  v.kind = std::get<0>(f);
  v.n = std::get<1>(f);
  v.shift = std::get<2>(f);
  v.fast_rho = std::get<3>(f);
  v.inv_stat = std::get<4>(f);
  v.bounded_scores = std::get<5>(f);
  v.precise_output = std::get<6>(f);
  v.clamp = (float)std::get<7>(f);
  v.poly_rho = std::get<8>(f);
  return v;
}

PlanPtr flash_plan(const VariantFields& low, const std::optional<VariantFields>& high, double scale,
                   double bound, double vmax) {
  auto p = c10::make_intrusive<FlashPlan>();
  p->low = variant(low);
  p->guarded = high.has_value();
  if (p->guarded) p->high = variant(*high);
  p->scale = scale;
  p->bound = bound;
  p->vmax = vmax;
  return p;
}

// Custom VJP of flash.py:708-729 (residuals q_s, k, v, sink, o, stat). `sink`
// holds one logit per head, in units of `unit`; need_grad: a backward follows,
// whose workspace the forward prepares.
struct Flash : Function<Flash> {
  static Tensor forward(AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const std::optional<Tensor>& sink, double unit, const PlanPtr& plan,
                        bool need_grad) {
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3);
    Tensor guard, ws, bws, o_precise, s;
    if (sink.has_value()) s = sink->reshape({-1}).contiguous();
    if (plan->guarded) {
      guard = at::empty({algx_attn_guard_words()}, q.options().dtype(at::kInt));
      ws = scratch(algx_attn_forward_workspace_bytes(B, H, T, D), q);
    }
    Tensor q_s = at::empty_like(q), o = at::empty_like(q), stat = f32({B, H, T}, q);
    if (plan->precise()) o_precise = f32(q.sizes(), q);
    if (need_grad) bws = scratch(algx_attn_bwd_workspace_bytes(B, H, T, D), q);
    check(algx_attn_forward_unit(ptr(q), ptr(k), ptr(v), fptr(s), unit, ptr(q_s), ptr(o),
                                 fptr(o_precise), fptr(stat), static_cast<int32_t*>(ptr(guard)),
                                 ptr(ws), ptr(bws), B, H, T, D, dtype_code(q), plan->scale,
                                 plan->bound, plan->vmax, &plan->low, plan->hi(), stream()),
          "algx_attn_forward");
    ctx->save_for_backward({q_s, k, v, s, o, o_precise, stat, guard});
    ctx->saved_data["plan"] = at::IValue::make_capsule(plan);
    ctx->saved_data["unit"] = unit;
    if (sink.has_value()) ctx->saved_data["sink_shape"] = sink->sizes().vec();
    if (bws.defined()) ctx->saved_data["bws"] = bws;
    return o;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q_s = saved[0], &k = saved[1], &v = saved[2], &s = saved[3], &o = saved[4],
                 &o_precise = saved[5], &stat = saved[6], &guard = saved[7];
    const auto capsule = ctx->saved_data["plan"].toCapsule();
    const auto* plan = static_cast<const FlashPlan*>(capsule.get());
    const int64_t B = q_s.size(0), H = q_s.size(1), T = q_s.size(2), D = q_s.size(3);
    const Tensor dout = grad_like(grads[0], q_s);
    Tensor dq = at::empty_like(q_s), dk = at::empty_like(k), dv = at::empty_like(v), dsink;
    if (s.defined()) dsink = f32({H}, q_s);
    // The forward's prepared workspace serves one backward; a second one
    // (retain_graph) hands it over as raw memory.
    Tensor ws;
    int32_t state = ALGX_ATTN_WS_CLEARED;
    const auto kept = ctx->saved_data.find("bws");
    if (kept != ctx->saved_data.end()) {
      ws = kept->second.toTensor();
      ctx->saved_data.erase(kept);
    } else {
      ws = scratch(algx_attn_bwd_workspace_bytes(B, H, T, D), q_s);
      state = ALGX_ATTN_WS_RAW;
    }
    check(algx_attn_bwd_unit(ptr(q_s), ptr(k), ptr(v), fptr(s), ctx->saved_data["unit"].toDouble(),
                             ptr(o), fptr(o_precise), fptr(stat), ptr(dout), ptr(dq), ptr(dk),
                             ptr(dv), fptr(dsink), ptr(ws), state, B, H, T, D, dtype_code(q_s),
                             plan->scale, &plan->low, plan->hi(),
                             static_cast<const int32_t*>(ptr(guard)), stream()),
          "algx_attn_bwd");
    if (dsink.defined()) dsink = dsink.reshape(ctx->saved_data["sink_shape"].toIntVector());
    return {dq, dk, dv, dsink, Tensor(), Tensor(), Tensor()};
  }
};

Tensor flash(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& sink,
             double unit, const PlanPtr& plan) {
  on_device(q, "flash_attention");
  const bool need = at::GradMode::is_enabled() &&
                    (q.requires_grad() || k.requires_grad() || v.requires_grad() ||
                     (sink.has_value() && sink->requires_grad()));
  return Flash::apply(q.contiguous(), k.contiguous(), v.contiguous(), sink, unit, plan, need);
}

// ---------------------------------------------------------------- fused head

// Custom VJP of fused_head.py:232-257 (residuals h, E, targets, stat).
struct Head : Function<Head> {
  static variable_list forward(AutogradContext* ctx, const Tensor& h, const Tensor& embed,
                               const Tensor& targets, int64_t kind, int64_t n, double c,
                               double clamp) {
    const int64_t N = h.size(0), d = h.size(1), V = embed.size(0);
    const Tensor e = embed.to(h.scalar_type()).contiguous();  // fused_head.py:168
    Tensor stat = f32({N}, h), tel = f32({N}, h), obj = f32({}, h);
    const int32_t dt = dtype_code(h);
    Tensor ws = scratch(algx_head_loss_workspace_bytes(N, d, V, dt), h);
    check(algx_head_loss(ptr(h), ptr(e), static_cast<const int32_t*>(ptr(targets)), fptr(stat),
                         fptr(tel), fptr(obj), ptr(ws), N, d, V, kind, n, (float)(1.0 / c),
                         (float)clamp, dt, stream()),
          "algx_head_loss");
    ctx->save_for_backward({h, e, targets, stat});
    ctx->saved_data["kind"] = kind;
    ctx->saved_data["n"] = n;
    ctx->saved_data["c"] = c;
    ctx->saved_data["clamp"] = clamp;
    ctx->saved_data["embed"] = embed.scalar_type();
    ctx->mark_non_differentiable({tel});
    return {obj, tel};
  }

  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &h = saved[0], &e = saved[1], &targets = saved[2], &stat = saved[3];
    const int64_t kind = ctx->saved_data["kind"].toInt(), n = ctx->saved_data["n"].toInt();
    const double c = ctx->saved_data["c"].toDouble(), clamp = ctx->saved_data["clamp"].toDouble();
    const int64_t N = h.size(0), d = h.size(1), V = e.size(0);
    const int32_t dt = dtype_code(h);
    const double slope = kind == ALGX_HEAD_CE ? 1.0 : n / c;
    const Tensor scale = grads[0].to(at::kFloat).mul(slope / N).reshape({1}).contiguous();
    Tensor dh = at::empty_like(h), de = f32({V, d}, h);
    Tensor ws = scratch(algx_head_bwd_workspace_bytes(N, d, V, dt), h);
    check(algx_head_bwd(ptr(h), ptr(e), static_cast<const int32_t*>(ptr(targets)), fptr(stat),
                        fptr(scale), ptr(dh), fptr(de), ptr(ws), N, d, V, kind, n,
                        (float)(1.0 / c), (float)clamp, dt, stream()),
          "algx_head_bwd");
    const auto embed = static_cast<at::ScalarType>(ctx->saved_data["embed"].toInt());
    return {dh, de.to(embed), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor> head(const Tensor& h, const Tensor& embed, const Tensor& targets,
                                int64_t kind, int64_t n, double c, double clamp) {
  on_device(h, "fused_head");
  const Tensor t32 = targets.to(h.options().dtype(at::kInt).requires_grad(false)).contiguous();
  const variable_list out = Head::apply(h.contiguous(), embed, t32, kind, n, c, clamp);
  return {out[0], out[1]};
}

// ------------------------------------------------------------------- QK-norm

// rms_norm of D = 64 rows with a gain, of one tensor or of the attention's q
// and k in one launch each way (native VJP, qk_norm.py:29-59).
struct QkNorm : Function<QkNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& gain, double eps) {
    Tensor y = at::empty_like(x);
    check(algx_qknorm_fwd(ptr(x), fptr(gain), ptr(y), x.numel() / 64, 64, dtype_code(x), eps,
                          stream()),
          "algx_qknorm_fwd");
    ctx->save_for_backward({x, gain});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &gain = saved[1];
    const int64_t rows = x.numel() / 64;
    const int32_t dt = dtype_code(x);
    const Tensor dy = grad_like(grads[0], x);
    Tensor dx = at::empty_like(x), dgain = f32({64}, x);
    Tensor ws = scratch(algx_qknorm_bwd_workspace_bytes(rows, 64, dt), x);
    check(algx_qknorm_bwd(ptr(x), fptr(gain), ptr(dy), ptr(dx), fptr(dgain), ptr(ws), rows, 64, dt,
                          ctx->saved_data["eps"].toDouble(), stream()),
          "algx_qknorm_bwd");
    return {dx, dgain, Tensor()};
  }
};

struct QkNormPair : Function<QkNormPair> {
  static variable_list forward(AutogradContext* ctx, const Tensor& q, const Tensor& k,
                               const Tensor& gain_q, const Tensor& gain_k, double eps) {
    Tensor yq = at::empty_like(q), yk = at::empty_like(k);
    check(algx_qknorm_pair_fwd(ptr(q), ptr(k), fptr(gain_q), fptr(gain_k), ptr(yq), ptr(yk),
                               q.numel() / 64, 64, dtype_code(q), eps, stream()),
          "algx_qknorm_pair_fwd");
    ctx->save_for_backward({q, k, gain_q, gain_k});
    ctx->saved_data["eps"] = eps;
    return {yq, yk};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &q = saved[0], &k = saved[1], &gain_q = saved[2], &gain_k = saved[3];
    const int64_t rows = q.numel() / 64;
    const int32_t dt = dtype_code(q);
    const Tensor dyq = grad_like(grads[0], q), dyk = grad_like(grads[1], k);
    Tensor dxq = at::empty_like(q), dxk = at::empty_like(k);
    Tensor dgq = f32({64}, q), dgk = f32({64}, q);
    Tensor ws = scratch(algx_qknorm_pair_bwd_workspace_bytes(rows, 64, dt), q);
    check(algx_qknorm_pair_bwd(ptr(q), ptr(k), fptr(gain_q), fptr(gain_k), ptr(dyq), ptr(dyk),
                               ptr(dxq), ptr(dxk), fptr(dgq), fptr(dgk), ptr(ws), rows, 64, dt,
                               ctx->saved_data["eps"].toDouble(), stream()),
          "algx_qknorm_pair_bwd");
    return {dxq, dxk, dgq, dgk, Tensor()};
  }
};

Tensor qk_norm(const Tensor& x, const Tensor& gain, double eps) {
  on_device(x, "qk_rms_norm");
  return QkNorm::apply(x.contiguous(), gain.contiguous(), eps);
}

std::tuple<Tensor, Tensor> qk_norm_pair(const Tensor& q, const Tensor& k, const Tensor& gain_q,
                                        const Tensor& gain_k, double eps) {
  on_device(q, "qk_rms_norm_pair");
  const variable_list y = QkNormPair::apply(q.contiguous(), k.contiguous(), gain_q.contiguous(),
                                            gain_k.contiguous(), eps);
  return {y[0], y[1]};
}

// ------------------------------------------------- norms and gated products

struct RmsNorm : Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const std::optional<Tensor>& gain,
                        double eps) {
    const Tensor g = gain.value_or(Tensor());
    Tensor y = at::empty_like(x);
    check(algx_rms_norm_fwd(ptr(x), fptr(g), ptr(y), rows_of(x), x.size(-1), dtype_code(x), eps,
                            stream()),
          "algx_rms_norm_fwd");
    ctx->save_for_backward({x, g});
    ctx->saved_data["eps"] = eps;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &gain = saved[1];
    const int64_t rows = rows_of(x), D = x.size(-1);
    const int32_t dt = dtype_code(x);
    const Tensor dy = aligned_grad(grads[0], x);
    Tensor dx = at::empty_like(x), dgain, ws;
    if (gain.defined()) {
      dgain = f32({D}, x);
      ws = scratch(algx_rms_norm_bwd_workspace_bytes(rows, D, dt), x);
    }
    check(algx_rms_norm_bwd(ptr(x), fptr(gain), ptr(dy), ptr(dx), fptr(dgain), ptr(ws), rows, D,
                            dt, ctx->saved_data["eps"].toDouble(), stream()),
          "algx_rms_norm_bwd");
    return {dx, dgain, Tensor()};
  }
};

struct AddRmsNorm : Function<AddRmsNorm> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& r,
                               const std::optional<Tensor>& gain, double eps) {
    const Tensor g = gain.value_or(Tensor());
    Tensor xsum = at::empty_like(x), y = at::empty_like(x);
    check(algx_add_rms_norm_fwd(ptr(x), ptr(r), fptr(g), ptr(xsum), ptr(y), rows_of(x), x.size(-1),
                                dtype_code(x), eps, stream()),
          "algx_add_rms_norm_fwd");
    ctx->save_for_backward({xsum, g});
    ctx->saved_data["eps"] = eps;
    return {xsum, y};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &xsum = saved[0], &gain = saved[1];
    const int64_t rows = rows_of(xsum), D = xsum.size(-1);
    const int32_t dt = dtype_code(xsum);
    const Tensor dres = aligned_grad(grads[0], xsum), dy = aligned_grad(grads[1], xsum);
    Tensor dx = at::empty_like(xsum), dgain, ws;
    if (gain.defined()) {
      dgain = f32({D}, xsum);
      ws = scratch(algx_rms_norm_bwd_workspace_bytes(rows, D, dt), xsum);
    }
    check(algx_add_rms_norm_bwd(ptr(xsum), fptr(gain), ptr(dy), ptr(dres), ptr(dx), fptr(dgain),
                                ptr(ws), rows, D, dt, ctx->saved_data["eps"].toDouble(), stream()),
          "algx_add_rms_norm_bwd");
    return {dx, dx, dgain, Tensor()};
  }
};

struct GluPacked : Function<GluPacked> {
  static Tensor forward(AutogradContext* ctx, const Tensor& gu, int64_t act, double beta) {
    const int64_t cols = gu.size(-1) / 2, rows = gu.numel() / (2 * cols);
    std::vector<int64_t> shape = gu.sizes().vec();
    shape.back() = cols;
    Tensor y = at::empty(shape, gu.options());
    check(algx_glu_packed_fwd(ptr(gu), ptr(y), rows, cols, act, dtype_code(gu), beta, stream()),
          "algx_glu_packed_fwd");
    ctx->save_for_backward({gu});
    ctx->saved_data["act"] = act;
    ctx->saved_data["beta"] = beta;
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor gu = ctx->get_saved_variables()[0];
    const int64_t cols = gu.size(-1) / 2, rows = gu.numel() / (2 * cols);
    const Tensor dy = aligned(grads[0].to(gu.scalar_type()));
    Tensor dgu = at::empty_like(gu);
    check(algx_glu_packed_bwd(ptr(gu), ptr(dy), ptr(dgu), rows, cols,
                              ctx->saved_data["act"].toInt(), dtype_code(gu),
                              ctx->saved_data["beta"].toDouble(), stream()),
          "algx_glu_packed_bwd");
    return {dgu, Tensor(), Tensor()};
  }
};

Tensor rms_norm(const Tensor& x, const std::optional<Tensor>& gain, double eps) {
  on_device(x, "rms_norm");
  return RmsNorm::apply(aligned(x), opt(gain32(gain)), eps);
}

std::tuple<Tensor, Tensor> add_rms_norm(const Tensor& x, const Tensor& r,
                                        const std::optional<Tensor>& gain, double eps) {
  on_device(x, "add_rms_norm");
  const variable_list out = AddRmsNorm::apply(aligned(x), aligned(r), opt(gain32(gain)), eps);
  return {out[0], out[1]};
}

Tensor glu_packed(const Tensor& gu, int64_t act, double beta) {
  TORCH_CHECK_VALUE(gu.size(-1) >= 2, "glu_packed needs a gate and an up column at least");
  on_device(gu, "glu_packed");
  return GluPacked::apply(aligned(gu), act, beta);
}

// ------------------------------------------- prologue, layout, projection

// Projections -> attention inputs (model.py:166-174) and the VJP.
struct Prologue : Function<Prologue> {
  static variable_list forward(AutogradContext* ctx, const Tensor& qkv,
                               const std::optional<Tensor>& q_gain,
                               const std::optional<Tensor>& k_gain,
                               const std::optional<Tensor>& cos, const std::optional<Tensor>& sin,
                               int64_t H, double eps) {
    const int64_t B = qkv.size(0), T = qkv.size(1), three_d = qkv.size(2), d = three_d / 3;
    const Tensor qg = q_gain.value_or(Tensor()), kg = k_gain.value_or(Tensor());
    const Tensor ct = cos.value_or(Tensor()), st = sin.value_or(Tensor());
    variable_list out(3);
    for (auto& t : out) t = at::empty({B, H, T, d / H}, qkv.options());
    const char* base = static_cast<const char*>(ptr(qkv));
    const int64_t step = d * qkv.element_size();
    check(algx_qk_prologue_fwd(base, base + step, base + 2 * step, three_d, fptr(qg), fptr(kg),
                               fptr(ct), fptr(st), ptr(out[0]), ptr(out[1]), ptr(out[2]), B, T, H,
                               d / H, dtype_code(qkv), eps, stream()),
          "algx_qk_prologue_fwd");
    ctx->save_for_backward({qkv, qg, kg, ct, st});
    ctx->saved_data["H"] = H;
    ctx->saved_data["eps"] = eps;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &qkv = saved[0], &qg = saved[1], &kg = saved[2], &ct = saved[3], &st = saved[4];
    const int64_t H = ctx->saved_data["H"].toInt();
    const int64_t B = qkv.size(0), T = qkv.size(1), three_d = qkv.size(2), d = three_d / 3;
    const int32_t dt = dtype_code(qkv);
    Tensor g[3];
    for (int i = 0; i < 3; ++i)
      g[i] = grads[i].defined() ? grads[i].to(qkv.scalar_type()).contiguous()
                                : at::zeros({B, H, T, d / H}, qkv.options());
    Tensor dqkv = at::empty_like(qkv), dqg, dkg, ws;
    if (qg.defined()) {
      dqg = f32({d / H}, qkv);
      dkg = f32({d / H}, qkv);
      ws = scratch(algx_qk_prologue_bwd_workspace_bytes(B, T, H, d / H, dt), qkv);
    }
    const char* in = static_cast<const char*>(ptr(qkv));
    char* base = static_cast<char*>(ptr(dqkv));
    const int64_t step = d * qkv.element_size();
    check(algx_qk_prologue_bwd(in, in + step, fptr(qg), fptr(kg), fptr(ct), fptr(st), ptr(g[0]),
                               ptr(g[1]), ptr(g[2]), base, base + step, base + 2 * step, three_d,
                               fptr(dqg), fptr(dkg), ptr(ws), B, T, H, d / H, dt,
                               ctx->saved_data["eps"].toDouble(), stream()),
          "algx_qk_prologue_bwd");
    return {dqkv, dqg, dkg, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor, Tensor> prologue(const Tensor& qkv, const std::optional<Tensor>& q_gain,
                                            const std::optional<Tensor>& k_gain,
                                            const std::optional<Tensor>& cos,
                                            const std::optional<Tensor>& sin, int64_t H,
                                            double eps) {
  TORCH_CHECK_VALUE(H > 0, "attention_prologue needs one head at least");
  on_device(qkv, "attention_prologue");
  const variable_list out = Prologue::apply(qkv.contiguous(), opt(gain32(q_gain)),
                                            opt(gain32(k_gain)), cos, sin, H, eps);
  return {out[0], out[1], out[2]};
}

// (B, P, Q, row) -> (B, Q, P, row) as a new tensor.
Tensor swap(const Tensor& x, int64_t B, int64_t P, int64_t Q, int64_t row) {
  const Tensor in = aligned(x);
  Tensor out = at::empty({B, Q, P, row}, in.options());
  check(algx_swap_axes(ptr(in), ptr(out), B, P, Q, row * in.element_size(), stream()),
        "algx_swap_axes");
  return out;
}

struct HeadsToTokens : Function<HeadsToTokens> {
  static Tensor forward(AutogradContext* ctx, const Tensor& a) {
    const int64_t B = a.size(0), H = a.size(1), T = a.size(2), D = a.size(3);
    ctx->saved_data["shape"] = a.sizes().vec();
    const Tensor in = aligned(a);
    Tensor out = at::empty({B, T, H * D}, in.options());
    check(algx_swap_axes(ptr(in), ptr(out), B, H, T, D * in.element_size(), stream()),
          "algx_swap_axes");
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto s = ctx->saved_data["shape"].toIntVector();
    return {swap(grads[0], s[0], s[2], s[1], s[3])};
  }
};

Tensor heads_to_tokens(const Tensor& a) {
  on_device(a, "heads_to_tokens");
  return HeadsToTokens::apply(a);
}

// x^T g in bf16 for x (T, din), g (T, dout): float32 sums of chunks of T added
// in chunk order.
Tensor weight_grad(const Tensor& x, const Tensor& g) {
  TORCH_CHECK_VALUE(x.dim() == 2 && g.dim() == 2 && g.size(0) >= x.size(0),
                    "weight_grad needs (T, din) inputs and (T, dout) gradients");
  const Tensor x2 = aligned(x), g2 = aligned(g);
  const int64_t T = x2.size(0), din = x2.size(1), dout = g2.size(1);
  Tensor ws = scratch(algx_weight_grad_workspace_bytes(T, din, dout), x2);
  Tensor out = at::empty({din, dout}, x2.options());
  check(algx_weight_grad(ptr(x2), ptr(g2), ptr(out), ptr(ws), T, din, dout, stream()),
        "algx_weight_grad");
  return out;
}

struct Project : Function<Project> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w) {
    ctx->save_for_backward({x, w});
    return at::matmul(x, w);
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const variable_list saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1];
    const int64_t din = w.size(0), dout = w.size(1);
    const Tensor g = grads[0].contiguous();
    Tensor dx, dw;
    if (ctx->needs_input_grad(0)) dx = at::matmul(g, w.t());
    if (ctx->needs_input_grad(1))
      dw = weight_grad(x.reshape({-1, din}), g.reshape({-1, dout}));
    return {dx, dw};
  }
};

Tensor project(const Tensor& x, const Tensor& w) { return Project::apply(x, w); }

}  // namespace

PYBIND11_MODULE(_ops, m) {
  // The interpreter lock is released while a call runs, as for a ctypes call.
  typedef py::call_guard<py::gil_scoped_release> nogil;
  py::class_<FlashPlan, PlanPtr>(m, "FlashPlan");
  m.def("flash_plan", &flash_plan);
  m.def("flash", &flash, nogil());
  m.def("head", &head, nogil());
  m.def("qk_norm", &qk_norm, nogil());
  m.def("qk_norm_pair", &qk_norm_pair, nogil());
  m.def("rms_norm", &rms_norm, nogil());
  m.def("add_rms_norm", &add_rms_norm, nogil());
  m.def("glu_packed", &glu_packed, nogil());
  m.def("prologue", &prologue, nogil());
  m.def("heads_to_tokens", &heads_to_tokens, nogil());
  m.def("weight_grad", &weight_grad, nogil());
  m.def("project", &project, nogil());
}
