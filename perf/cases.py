"""Workloads for timing the framework through its public entry points.

``listed()`` names the fixed cases, ``draw(rng)`` one more of the same ranges.
A case is a dict of plain values; ``kind`` picks the entry point:

* ``attention``: ``kernels.flash_attention`` on (B, H, T, 64), forward alone
  (``grad=False``) or forward and backward, the asinh-power weights behind the
  range guard as the model calls them, or the softmax arm;
* ``head``: ``kernels.fused_head``, objective, telemetry and both gradients,
  from a float32 embedding as the model keeps it;
* ``qk_norm``: ``kernels.qk_rms_norm_pair``, forward and backward;
* ``ffn``: the block's residual norm and gated product,
  ``algebraic.add_rms_norm`` and ``algebraic.glu_packed``, both ways;
* ``muon``: ``optimizers.newton_schulz_many`` over a model's layer matrices;
* ``model``: ``model.train_objective`` and the gradient of every parameter.

``exact(case, seed)`` is the same result in float64 from plain torch.
"""

import math
import os
import sys

import torch
import torch.utils.checkpoint

# The package sits one folder below the repository's root (the working folder).
_PKG = os.path.join(os.getcwd(), "algebraic-extra_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from algebraic_amd import config, model, optimizers  # noqa: E402
from algebraic_amd.algebraic import add_rms_norm, glu_packed  # noqa: E402
from algebraic_amd.kernels import flash_attention, fused_head, qk_rms_norm_pair  # noqa: E402

DEV = "cuda"
D = 64                      # head width of every preset
EPS = 1e-5
SIZES = {"proxy": (384, 8, 6, 1024), "125m": (768, 12, 12, 2048), "350m": (1024, 24, 16, 2688)}
DT = {"bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # The smallest call: the float32 forward of BASELINE's first
        # configuration, a check of one short sequence. Launches and host time.
        dict(name="attn_f32_short", kind="attention", weights="asinh", dtype="f32", B=1, H=4,
             T=256, sink=False, grad=False),
        # Fine-tuning on a document whose length is what it is (any T up to
        # 512 is accepted as it stands).
        dict(name="attn_ragged", kind="attention", weights="asinh", dtype="bf16", B=2, H=12,
             T=333, sink=True, grad=True),
        # The comparison arm at the proxy size's width and default length.
        dict(name="attn_proxy_softmax", kind="attention", weights="softmax", dtype="bf16", B=8,
             H=6, T=1024, sink=False, grad=True),
        # The headline attention: one layer of the 350M training step.
        dict(name="attn_350m", kind="attention", weights="asinh", dtype="bf16", B=8, H=16,
             T=2048, sink=True, grad=True),
        # The head of one default-length sequence of the proxy model.
        dict(name="head_proxy_ce", kind="head", loss="ce", dtype="bf16", N=1024, d=384, V=32768),
        # The headline head: 8 x 2048 tokens against the 50304-word vocabulary.
        dict(name="head_125m", kind="head", loss="alg_ce", dtype="bf16", N=16384, d=768, V=50304),
        # The same head of a float32 model, one sequence.
        dict(name="head_f32", kind="head", loss="alg_ce", dtype="f32", N=1024, d=384, V=32768),
        # The headline QK-norm: q and k of one 350M layer.
        dict(name="qk_norm_350m", kind="qk_norm", dtype="bf16", B=8, T=2048, H=16),
        # Residual norm and gated product of one 350M block.
        dict(name="ffn_350m", kind="ffn", dtype="bf16", act="alu", rows=16384, d=1024, ff=2688),
        # Muon's orthogonalisation for the 125M model's layers.
        dict(name="muon_125m", kind="muon", size="125m", layers=12),
        # A training step of the smallest model on little data.
        dict(name="model_proxy", kind="model", preset="algebraic", size="proxy", B=2, T=512,
             V=32768),
        # The headline model: a 350M training step, 8 x 2048 tokens.
        dict(name="model_350m", kind="model", preset="algebraic", size="350m", B=8, T=2048,
             V=50304),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("attention", "head", "qk_norm", "ffn", "muon", "model"),
                       weights=(9, 6, 2, 2, 2, 2))[0]
    if kind == "attention":
        dtype = "bf16" if rng.random() < 0.8 else "f32"
        T = _log(rng, 48, 4096)
        if rng.random() < 0.5:
            T = max(128, T // 128 * 128)
        if dtype == "f32" or T % 128:
            T = min(T, 1023)
        B, H = rng.randint(1, 8), rng.choice((4, 6, 12, 16, 24))
        limit = 2.0e9 if dtype == "f32" or T % 128 else 3.5e10      # flops of one head's product
        while B > 1 and 2.0 * B * H * T * T * D > limit:
            B -= 1
        return dict(kind=kind, weights=rng.choice(("asinh", "asinh", "softmax")), dtype=dtype,
                    B=B, H=H, T=T, sink=rng.random() < 0.5, grad=rng.random() < 0.7)
    if kind == "head":
        dtype = "bf16" if rng.random() < 0.8 else "f32"
        top = 16384 if dtype == "bf16" else 1024
        N = _log(rng, 32, top)
        N = N if N < 128 else N // 128 * 128        # whole token blocks, as the entry point asks
        V = _log(rng, 1000, 60000)
        V = V // 128 * 128 if rng.random() < 0.4 else V
        return dict(kind=kind, loss=rng.choice(("ce", "alg_ce")), dtype=dtype, N=N,
                    d=rng.choice((384, 768, 1024, 1536) if dtype == "bf16" else (384, 768)), V=V)
    if kind == "qk_norm":
        B, H = rng.randint(1, 8), rng.choice((4, 6, 12, 16, 24))
        return dict(kind=kind, dtype="bf16" if rng.random() < 0.8 else "f32", B=B,
                    T=8 * _log(rng, 8, 256) + 8 * rng.randint(0, 3), H=H)
    if kind == "ffn":
        return dict(kind=kind, dtype="bf16" if rng.random() < 0.8 else "f32",
                    act=rng.choice(("alu", "silu")), rows=_log(rng, 64, 16384),
                    d=64 * rng.randint(3, 24), ff=8 * rng.randint(48, 528))
    if kind == "muon":
        size = rng.choice(("proxy", "125m", "350m"))
        return dict(kind=kind, size=size, layers=rng.randint(1, 8))
    T = rng.randint(64, 512)
    return dict(kind=kind, preset=rng.choice(("standard", "algebraic")),
                size=rng.choice(("proxy", "125m")), B=rng.randint(1, 4),
                T=T // 64 * 64 if rng.random() < 0.6 else T, V=rng.choice((32768, 50304)))


# ------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _unit(x):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)


def _attention_inputs(case, seed):
    """QK-normed queries and keys, values and output gradient ~ N(0, 1)."""
    g, dt = _gen(seed), DT[case["dtype"]]
    shape = (case["B"], case["H"], case["T"], D)
    q, k = _unit(_randn(g, *shape)).to(dt), _unit(_randn(g, *shape)).to(dt)
    v, do = _randn(g, *shape).to(dt), _randn(g, *shape).to(dt)
    sink = 0.5 * _randn(g, case["H"]) if case["sink"] else None
    return q, k, v, sink, do


def _head_inputs(case, seed):
    """Normalised hidden states, a float32 embedding at init_std, random targets."""
    g = _gen(seed)
    h = _unit(_randn(g, case["N"], case["d"])).to(DT[case["dtype"]])
    e = 0.02 * _randn(g, case["V"], case["d"])
    t = torch.randint(0, case["V"], (case["N"],), generator=g, device=DEV)
    return h, e, t


def _qk_inputs(case, seed):
    g, dt = _gen(seed), DT[case["dtype"]]
    shape = (case["B"], case["T"], case["H"], D)
    x = [_randn(g, *shape).to(dt) for _ in range(4)]
    gains = [1.0 + 0.01 * _randn(g, D) for _ in range(2)]
    return x[0], x[1], gains[0], gains[1], x[2], x[3]


def _ffn_inputs(case, seed):
    g, dt = _gen(seed), DT[case["dtype"]]
    rows, d, ff = case["rows"], case["d"], case["ff"]
    x, r, ds, dy = (_randn(g, rows, d).to(dt) for _ in range(4))
    gain = 1.0 + 0.05 * _randn(g, d)
    gu, dp = _randn(g, rows, 2 * ff).to(dt), _randn(g, rows, ff).to(dt)
    return x, r, gain, ds, dy, gu, dp


def _muon_inputs(case, seed):
    """Momentum look-aheads of the stacked weights: w_q, w_k, w_v, w_o, w_g, w_u, w_d."""
    g, L = _gen(seed), case["layers"]
    d, _, _, f = SIZES[case["size"]]
    return [1e-3 * _randn(g, L, a, b) for a, b in ((d, d),) * 4 + ((d, f), (d, f), (f, d))]


def _model_inputs(case, seed):
    """Parameters at their initial statistics, random tokens and targets."""
    g = _gen(seed)
    d, L, H, f = SIZES[case["size"]]
    V = case["V"]

    def w(*shape):
        return 0.02 * _randn(g, *shape)

    layers = {"w_q": w(L, d, d), "w_k": w(L, d, d), "w_v": w(L, d, d), "w_o": w(L, d, d),
              "w_g": w(L, d, f), "w_u": w(L, d, f), "w_d": w(L, f, d),
              "ln1": torch.ones(L, d, device=DEV), "ln2": torch.ones(L, d, device=DEV)}
    if case["preset"] == "algebraic":
        layers["q_gain"] = torch.ones(L, D, device=DEV)
        layers["k_gain"] = torch.ones(L, D, device=DEV)
        layers["sink"] = torch.zeros(L, H, device=DEV)
    params = {"embed": w(V, d), "embed_gain": torch.ones(d, device=DEV),
              "final_gain": torch.ones(d, device=DEV), "layers": layers}
    tok = torch.randint(0, V, (2, case["B"], case["T"]), generator=g, device=DEV)
    return params, tok[0], tok[1]


def _leaves(params):
    out = [params[n] for n in ("embed", "embed_gain", "final_gain")]
    return out + list(params["layers"].values())


# ------------------------------------------------------------- prepare, run

def prepare(case, seed):
    kind = case["kind"]
    if kind == "attention":
        q, k, v, sink, do = _attention_inputs(case, seed)
        leaves = [t.requires_grad_(case["grad"]) for t in (q, k, v, sink) if t is not None]
        kw = dict(kind=case["weights"], block=512 if case["T"] % 512 == 0 else case["T"])
        if case["weights"] == "asinh":
            kw.update(n=16, c=8.0, range_guard=True)
        return dict(case=case, leaves=leaves, do=do, kw=kw)
    if kind == "head":
        h, e, t = _head_inputs(case, seed)
        kw = dict(kind=case["loss"], n=8 if case["loss"] == "alg_ce" else 16,
                  c=2.0 if case["loss"] == "alg_ce" else 16.0)
        return dict(case=case, leaves=[h.requires_grad_(), e.requires_grad_()], targets=t, kw=kw)
    if kind == "qk_norm":
        q, k, gq, gk, dq, dk = _qk_inputs(case, seed)
        return dict(case=case, leaves=[t.requires_grad_() for t in (q, k, gq, gk)], dy=(dq, dk))
    if kind == "ffn":
        x, r, gain, ds, dy, gu, dp = _ffn_inputs(case, seed)
        return dict(case=case, leaves=[t.requires_grad_() for t in (x, r, gain, gu)],
                    dy=(ds, dy, dp))
    if kind == "muon":
        return dict(case=case, Gs=_muon_inputs(case, seed))
    params, tokens, targets = _model_inputs(case, seed)
    leaves = [t.requires_grad_() for t in _leaves(params)]
    cfg = config.build(case["preset"], case["size"], vocab_size=case["V"], seq_len=case["T"],
                       attn_impl="flash", head_impl="fused", remat=False,
                       flash_block=case["T"] if case["T"] % 512 else 512,
                       head_block_n=case["T"] if case["B"] * case["T"] % 128 else 128)
    return dict(case=case, params=params, leaves=leaves, tokens=tokens, targets=targets, cfg=cfg,
                tables=model.position_tables(cfg))


def run(state):
    kind = state["case"]["kind"]
    if kind == "attention":
        leaves, kw = state["leaves"], state["kw"]
        if not state["case"]["grad"]:
            with torch.no_grad():
                return flash_attention(*leaves, **kw)
        o = flash_attention(*leaves, **kw)
        return (o.detach(),) + torch.autograd.grad(o, leaves, state["do"])
    if kind == "head":
        h, e = state["leaves"]
        obj, tel = fused_head(h, e, state["targets"], **state["kw"])
        return (obj.detach(), tel) + torch.autograd.grad(obj, [h, e])
    if kind == "qk_norm":
        y = qk_rms_norm_pair(*state["leaves"], EPS, block=8)
        grads = torch.autograd.grad(y, state["leaves"], state["dy"])
        return tuple(t.detach() for t in y) + grads
    if kind == "ffn":
        x, r, gain, gu = state["leaves"]
        s, y = add_rms_norm(x, r, gain, EPS)
        p = glu_packed(gu, state["case"]["act"], 0.5)
        grads = torch.autograd.grad((s, y, p), (x, r, gain, gu), state["dy"])
        return (s.detach(), y.detach(), p.detach()) + grads
    if kind == "muon":
        return tuple(optimizers.newton_schulz_many(state["Gs"]))
    obj, tel = model.train_objective(state["params"], state["tokens"], state["targets"],
                                     state["cfg"], state["tables"])
    return (obj.detach(), tel) + torch.autograd.grad(obj, state["leaves"])


# ------------------------------------------------------------ work, tolerance

def work(case):
    kind = case["kind"]
    if kind in ("attention", "qk_norm", "ffn", "head"):
        es = 2 if case["dtype"] == "bf16" else 4
    if kind == "attention":
        n = case["B"] * case["H"] * case["T"] * D
        fwd = 2.0 * n * case["T"]               # two products over the causal half
        return {"bytes": es * n * (8 if case["grad"] else 4),
                "flops": fwd * (3.5 if case["grad"] else 1.0)}
    if kind == "head":
        N, d, V = case["N"], case["d"], case["V"]
        return {"bytes": 2 * es * N * d + 8.0 * V * d + 8 * N, "flops": 6.0 * N * d * V}
    if kind == "qk_norm":
        n = 2 * case["B"] * case["T"] * case["H"] * D
        return {"bytes": 5 * es * n, "flops": 16.0 * n}
    if kind == "ffn":
        rows, d, ff = case["rows"], case["d"], case["ff"]
        return {"bytes": es * rows * (8 * d + 6 * ff),
                "flops": rows * (16.0 * d + 30.0 * ff)}
    if kind == "muon":
        d, _, _, f = SIZES[case["size"]]
        # X X^T and A A are symmetric: half of each is enough.
        def flops(m, n):
            return 5 * (3.0 * m * m * n + m ** 3) + 2 * 3.0 * m * m * n
        L = case["layers"]
        return {"bytes": 8.0 * L * (4 * d * d + 3 * d * f),
                "flops": L * (4 * flops(d, d) + 3 * flops(d, f))}
    d, L, H, f = SIZES[case["size"]]
    V, tok = case["V"], case["B"] * case["T"]
    mats = L * (4 * d * d + 3 * d * f)
    return {"bytes": 8.0 * (mats + V * d),
            "flops": tok * (6.0 * (mats + V * d) + 7.0 * L * d * case["T"])}


def tolerance(case):
    """About four times the distance from float64 that each path shows: the
    rounding of its inputs' type and of the intermediates kept in it."""
    kind = case["kind"]
    if kind == "muon":
        return {"rel": 2.6e-2}      # seven bf16 products in a row: 6.6e-3
    if kind == "model":
        return {"rel": 1e-1}        # 8 to 24 bf16 layers: gradients 1e-2 .. 4e-2
    if case["dtype"] == "f32":
        return {"rel": 1.5e-5 if kind == "head" else 5e-6}      # dh 3.3e-6; 6e-7
    return {"rel": 7e-3 if kind == "qk_norm" else 1e-2}         # 1.7e-3; 2.0e-3 .. 3.2e-3


# ---------------------------------------------------------------- float64

F64 = torch.float64


def _attend64(q, k, v, sink, weights):
    """Causal attention by its logits: s / sqrt(D), or n asinh(s / (sqrt(D) c))."""
    s = q @ k.transpose(-1, -2) / math.sqrt(D)
    zs = None if sink is None else sink.reshape(1, -1, 1, 1)
    if weights == "asinh":
        s = 16.0 * torch.asinh(s / 8.0)
        zs = None if zs is None else 16.0 * torch.asinh(zs / 8.0)
    T = q.shape[-2]
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), -math.inf)
    if zs is None:
        return torch.softmax(s, -1) @ v
    s = torch.cat([s, zs.expand(s.shape[0], s.shape[1], T, 1)], -1)
    return torch.softmax(s, -1)[..., :T] @ v


def _norm64(x, gain):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gain


def _glu64(gu, act):
    gate, up = gu.chunk(2, -1)
    if act == "alu":
        u = 0.5 * up
        return gate * (0.5 * up * (1.0 + u * torch.rsqrt(1.0 + u * u)))
    return gate * up * torch.sigmoid(up)


def _head64(h, e, t, loss):
    """(objective, telemetry, the scalar whose gradient the entry point returns)."""
    z = h @ e.t()
    if loss == "alg_ce":
        z = 8.0 * torch.asinh(z / 2.0)
    nll = torch.logsumexp(z, -1) - z.gather(1, t[:, None])[:, 0]
    if loss == "ce":
        return nll.mean(), nll, nll.mean()
    p = torch.exp(-nll)
    return (1.0 - p).mean(), p, nll.mean()


def _model64(case, params, tokens, targets):
    d, L, H, f = SIZES[case["size"]]
    B, T = tokens.shape
    alg = case["preset"] == "algebraic"
    half = D // 2
    i = torch.arange(half, dtype=F64, device=DEV)
    theta = 10000.0 ** (-i / half)
    if alg:
        theta = 2.0 * torch.atan(0.5 * theta)           # ((1 + i w)^2 / (1 + w^2))^m
    ang = torch.arange(T, dtype=F64, device=DEV)[:, None] * theta
    cos, sin = torch.cos(ang), torch.sin(ang)

    def rotate(x):
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    def block(x, p):
        h = _norm64(x, p["ln1"])
        q, k, v = ((h @ p[n]).view(B, T, H, D).transpose(1, 2) for n in ("w_q", "w_k", "w_v"))
        if alg:
            q, k = _norm64(q, p["q_gain"]), _norm64(k, p["k_gain"])
        q, k = rotate(q), rotate(k)
        sink = p["sink"] if alg else None
        a = torch.cat([_attend64(q[b:b + 1], k[b:b + 1], v[b:b + 1], sink,
                                 "asinh" if alg else "softmax") for b in range(B)])
        x = x + a.transpose(1, 2).reshape(B, T, d) @ p["w_o"]
        h = _norm64(x, p["ln2"])
        gu = torch.cat([h @ p["w_g"], h @ p["w_u"]], -1)
        return x + _glu64(gu, "alu" if alg else "silu") @ p["w_d"]

    x = _norm64(params["embed"][tokens], params["embed_gain"])
    for l in range(L):
        p = {n: t[l] for n, t in params["layers"].items()}
        x = torch.utils.checkpoint.checkpoint(block, x, p, use_reentrant=False)
    h = _norm64(x, params["final_gain"]).reshape(B * T, d)
    return _head64(h, params["embed"], targets.reshape(-1), "alg_ce" if alg else "ce")


def _polar64(G):
    """The Muon iteration of optimizers.newton_schulz_5 on a stack of matrices."""
    M, N = G.shape[-2:]
    X = G.to(F64)
    X = X.transpose(-1, -2) if M > N else X
    X = X / torch.sqrt((X * X).sum((-2, -1), keepdim=True) + 1e-7)
    for _ in range(5):
        A = X @ X.transpose(-1, -2)
        X = 3.4445 * X + (-4.7750 * A + 2.0315 * (A @ A)) @ X
    for _ in range(2):
        X = 1.5 * X - 0.5 * (X @ X.transpose(-1, -2)) @ X
    X = X.transpose(-1, -2) if M > N else X
    return X * math.sqrt(max(1.0, M / N))


def exact(case, seed):
    kind = case["kind"]

    def up(*ts):
        return [None if t is None else t.to(F64).requires_grad_() for t in ts]

    if kind == "attention":
        q, k, v, sink, do = _attention_inputs(case, seed)
        outs = []
        (s64,) = up(sink)
        ds = 0.0
        for b in range(case["B"]):                       # one sequence at a time
            x = up(q[b:b + 1], k[b:b + 1], v[b:b + 1])
            o = _attend64(*x, s64, case["weights"])
            if not case["grad"]:
                outs.append((o.detach(),))
                continue
            leaves = x + ([] if s64 is None else [s64])
            g = torch.autograd.grad(o, leaves, do[b:b + 1].to(F64))
            outs.append((o.detach(),) + g[:3])
            ds = ds + g[3] if s64 is not None else ds
        full = tuple(torch.cat(t) for t in zip(*outs))
        if not case["grad"]:
            return full[0]
        return full + ((ds,) if s64 is not None else ())
    if kind == "head":
        h, e, t = _head_inputs(case, seed)
        h64, e64 = up(h, e.to(h.dtype))                  # the embedding is read in h's dtype
        obj, tel, loss = _head64(h64, e64, t, case["loss"])
        return (obj.detach(), tel.detach()) + torch.autograd.grad(loss, [h64, e64])
    if kind == "qk_norm":
        q, k, gq, gk, dq, dk = _qk_inputs(case, seed)
        x = up(q, k, gq, gk)
        y = (_norm64(x[0], x[2]), _norm64(x[1], x[3]))
        return tuple(t.detach() for t in y) + torch.autograd.grad(y, x, [dq.to(F64), dk.to(F64)])
    if kind == "ffn":
        x, r, gain, ds, dy, gu, dp = _ffn_inputs(case, seed)
        x, r, gain, gu = up(x, r, gain, gu)
        s = x + r
        y, p = _norm64(s, gain), _glu64(gu, case["act"])
        g = torch.autograd.grad((s, y, p), (x, r, gain, gu), [t.to(F64) for t in (ds, dy, dp)])
        return (s.detach(), y.detach(), p.detach()) + g
    if kind == "muon":
        return tuple(_polar64(G) for G in _muon_inputs(case, seed))
    params, tokens, targets = _model_inputs(case, seed)
    p64 = {n: t.to(F64).requires_grad_() for n, t in params.items() if n != "layers"}
    p64["layers"] = {n: t.to(F64).requires_grad_() for n, t in params["layers"].items()}
    obj, tel, loss = _model64(case, p64, tokens, targets)
    return (obj.detach(), tel.detach()) + torch.autograd.grad(loss, _leaves(p64))
