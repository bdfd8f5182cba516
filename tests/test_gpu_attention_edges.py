"""Attention at the edges of its kernels' blocks and tiles, against the oracle.

Tolerances as in tests/_tol.py; the sink gradient, a float32 sum over batch
and rows of terms formed from the storage dtype, as in test_gpu_attention.py.
"""

import math

import pytest
import torch

from _tol import rel_l2
from algebraic_amd import _lib
from algebraic_amd.kernels import flash_attention
from algebraic_amd.kernels.flash import _c_variant, make_variant
from test_gpu_attention import _check_all, _oracle, _rand, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("T", [1, 64, 127, 128, 129, 384])
def test_sink_gradient_row_blocks(T, dtype):
    """dsink is the sum of one share per pre-pass row block and sequence: one
    row, block edges of both dtypes (64 and 128 rows), several blocks, an odd
    head count and batch."""
    shape = (3, 5, T, 64)
    q, k, v, g = _rand(shape, 70 + T, dtype=dtype)
    sink = torch.tensor([0.4, -0.3, 0.0, 1.1, -0.8]).reshape(1, 5, 1, 1)
    kw = dict(kind="asinh", n=16, c=8.0, range_guard=True)
    got = _run(q, k, v, g, sink, block=T, **kw)
    want, _ = _oracle(q, k, v, g, sink, dtype, **kw)
    _check_all(got, want, dtype)


@pytest.mark.parametrize("T", [1, 2, 31, 33, 63, 65, 100, 127, 129, 191, 193, 255, 257, 333, 449])
@pytest.mark.parametrize("kw", [dict(kind="asinh", n=16, c=8.0, range_guard=True),
                                dict(kind="asinh", n=4, c=16.0, shift=True, fast_rho=True),
                                dict(kind="asinh", n=16, c=16.0, shift=False),
                                dict(kind="softmax")],
                         ids=["guarded", "shift", "clamped", "softmax"])
def test_mfma_any_length(T, kw):
    """bf16, D = 64 at lengths that end inside a wave's 32 rows, a 64-row tile,
    a 128-query or a 256-key block: rows past the end are read as row T - 1
    and must reach no output. Several heads, so that a write past one head
    would land in the next."""
    shape = (2, 3, T, 64)
    q, k, v, g = _rand(shape, 300 + T)
    sink = torch.tensor([0.3, -0.7, 0.1]).reshape(1, 3, 1, 1) if T % 2 else None
    got = _run(q, k, v, g, sink, block=T, **kw)
    want, _ = _oracle(q, k, v, g, sink, "bf16", **kw)
    _check_all(got, want, "bf16")


@pytest.mark.parametrize("T", [129, 300])
def test_mfma_any_length_out_of_range(T):
    """The guard's high variant at a ragged length: scores far outside the
    unshifted range, and a maximum that only the last row holds."""
    shape = (1, 2, T, 64)
    q, k, v, g = _rand(shape, 17)
    q[:, :, -1] *= 200.0
    k[:, :, -1] *= 200.0
    kw = dict(kind="asinh", n=16, c=8.0, range_guard=True)
    got = _run(q, k, v, g, None, block=T, **kw)
    want, res = _oracle(q, k, v, g, None, "bf16", **kw)
    _check_all(got, want, "bf16")


def test_ragged_backward_twice():
    """A second backward of one graph takes a raw workspace; dq needs nothing
    cleared at such a length."""
    q, k, v, g = (x.cuda().requires_grad_(True) for x in _rand((2, 3, 77, 64), 5))
    o = flash_attention(q, k, v, block=77, kind="asinh", n=16, c=8.0, range_guard=True)
    first = torch.autograd.grad(o, [q, k, v], g.detach(), retain_graph=True)
    second = torch.autograd.grad(o, [q, k, v], g.detach())
    for a, b in zip(first, second):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 63, 65, 130])
@pytest.mark.parametrize("kw", [dict(kind="asinh", n=16, c=8.0, range_guard=True),
                                dict(kind="asinh", n=8, c=1.0, shift=True, fast_rho=False),
                                dict(kind="softmax")], ids=["guarded", "shift", "softmax"])
def test_generic_row_tiles(T, D, dtype, kw):
    """The kernels for float32 and other head widths: one row, tile edges, fewer
    16-row tiles than waves and more, with and without a sink. (bf16 at
    D = 64 takes the bf16 MFMA kernels.)"""
    shape = (2, 2, T, D)
    q, k, v, g = _rand(shape, 500 + T + D, dtype=dtype)
    sink = torch.tensor([0.3, -0.7]).reshape(1, 2, 1, 1) if (T + D) % 2 else None
    got = _run(q, k, v, g, sink, block=T, **kw)
    want, _ = _oracle(q, k, v, g, sink, dtype, **kw)
    _check_all(got, want, dtype)


@pytest.mark.parametrize("kw", [dict(kind="asinh", n=16, c=8.0, shift=False),
                                dict(kind="softmax")], ids=["clamped", "softmax"])
def test_generic_later_rows_stay_apart(kw):
    """An infinity in a later row reaches no earlier one, also inside its
    16-row tile: o up to a value row, dv and dk from a query row onwards."""
    T, j = 40, 21
    q, k, v, g = (x.cuda() for x in _rand((1, 1, T, 64), 9, dtype="f32"))
    ref = [x.clone().requires_grad_() for x in (q, k, v)]
    o_ref = flash_attention(*ref, block=T, **kw)
    g_ref = torch.autograd.grad(o_ref, ref, g)
    bad = v.clone()
    bad[0, 0, j] = float("inf")
    o = flash_attention(q, k, bad, block=T, **kw)
    # such a tile is summed in another order: float32 rounding
    assert rel_l2(o[0, 0, :j], o_ref[0, 0, :j]) <= 1e-6
    assert not torch.isfinite(o[0, 0, j:]).any()
    bad = g.clone()
    bad[0, 0, j] = float("inf")
    o = flash_attention(*ref, block=T, **kw)
    dq, dk, dv = torch.autograd.grad(o, ref, bad)
    assert rel_l2(dq[0, 0, :j], g_ref[0][0, 0, :j]) <= 1e-6
    assert rel_l2(dv[0, 0, j + 1:], g_ref[2][0, 0, j + 1:]) <= 1e-6
    assert rel_l2(dk[0, 0, j + 1:], g_ref[1][0, 0, j + 1:]) <= 1e-6


@pytest.mark.parametrize("D,dtype", [(64, "f32"), (32, "f32"), (16, "bf16")])
@pytest.mark.parametrize("kw", [dict(kind="softmax"),
                                dict(kind="asinh", n=16, c=8.0, shift=True, fast_rho=False)],
                         ids=["softmax", "shift"])
def test_minus_infinite_scores(D, dtype, kw):
    """Scores of -inf (finite inputs whose product overflows) weigh nothing: a
    single key on the diagonal of a 16-row tile, a whole tile, a row's first
    tiles and all but one key. Such a row has no maximum yet where a wave meets
    nothing else first. Against float64, where the weights are exactly 0."""
    T, big = 130, 1e30
    pairs = {16: [16], 31: range(16, 32), 50: range(0, 16), 90: range(0, 90), 129: range(64, 130)}
    q, k, v, g = (x.cuda().float() for x in _rand((1, 1, T, D), 29, dtype="f32"))
    q[..., 0] = k[..., 0] = 0.0
    out = []
    for i, js in pairs.items():     # one query at a time: its keys hold the large value
        qi, ki = q.clone(), k.clone()
        qi[0, 0, i, 0] = -big
        ki[0, 0, list(js), 0] = big
        dt = torch.float32 if dtype == "f32" else torch.bfloat16
        leaves = [x.to(dt).requires_grad_() for x in (qi, ki, v)]
        o = flash_attention(*leaves, block=T, **kw)
        ref = [x.detach().double().requires_grad_() for x in leaves]
        s = ref[0] @ ref[1].transpose(-1, -2) / D ** 0.5
        if kw["kind"] == "asinh":
            s = kw["n"] * torch.asinh(s / kw["c"])
        p = torch.softmax(s.masked_fill(torch.ones(T, T, device=s.device).triu(1) > 0,
                                        -float("inf")), -1)
        want = p @ ref[2]
        tol = 1e-5 if dtype == "f32" else 1e-2      # float32 sums; bf16 weights and output
        assert torch.isfinite(o).all(), (i, js)
        assert rel_l2(o, want) <= tol, (i, js)
        if kw["kind"] == "softmax":
            got = torch.autograd.grad(o, leaves, g.to(dt))
            exp = torch.autograd.grad(want, ref, g.to(dt).double())
            for a, b, name in zip(got, exp, "qkv"):
                assert rel_l2(a[..., 1:], b[..., 1:]) <= (1e-4 if dtype == "f32" else 2e-2), name


def _abi(q, k, v, do, lo, hi=None, guard=None, entry="split", bounds=None):
    """o, dq, dk, dv of the C ABI calls for the given variants. Forward entry
    points: "split", prepare and forward, the guard word set by the caller; or
    one call that forms the word (expected to be `guard`; without `bounds`, by
    bounds that every input keeps or misses): "fused" with a workspace,
    "no_workspace" without one, "noalloc"."""
    B, H, T, D = q.shape
    dt, st, p = _lib.dtype_code(q.dtype), _lib.stream(), _lib.ptr
    scale = 1.0 / (8.0 * math.sqrt(D))
    bound, vmax = bounds or (1e9 if guard else 0.0, 1e9)
    q_s, o, dq, dk, dv = (torch.empty_like(q) for _ in range(5))
    o_precise = torch.empty(q.shape, dtype=torch.float32, device="cuda")
    stat = torch.empty((B, H, T), dtype=torch.float32, device="cuda")
    # NaN where the backward expects nothing cleared
    bws = torch.full((_lib.query("algx_attn_bwd_workspace_bytes", B, H, T, D) // 4,),
                     float("nan"), device="cuda")
    ws = word = None
    if entry == "fused":
        ws = torch.empty(_lib.query("algx_attn_forward_workspace_bytes", B, H, T, D),
                         dtype=torch.uint8, device="cuda")
    if guard is not None:
        word = torch.zeros(_lib.query("algx_attn_guard_words"), dtype=torch.int32, device="cuda")
        word[0] = guard if entry == "split" else 7
    outs = (p(q), p(k), p(v), None, p(q_s), p(o), p(o_precise), p(stat), p(word))
    tail = (p(bws), B, H, T, D, dt, scale, bound, vmax, lo, hi, st)
    if entry == "noalloc":
        _lib.call("algx_attn_forward_noalloc", *outs, *tail)
    elif entry != "split":
        _lib.call("algx_attn_forward", *outs, p(ws), *tail)
    else:
        _lib.call("algx_attn_prepare", p(q), p(k), p(v), None, p(q_s), None, B, H, T, D, dt, scale,
                  0.0, 0.0, st)
        _lib.call("algx_attn_fwd", p(q_s), p(k), p(v), None, p(o), p(o_precise), p(stat), B, H, T,
                  D, dt, lo, hi, p(word), st)
    state = _lib.ATTN_WS_RAW if entry == "split" else _lib.ATTN_WS_CLEARED
    _lib.call("algx_attn_bwd", p(q_s), p(k), p(v), None, p(o), p(o_precise), p(stat), p(do), p(dq),
              p(dk), p(dv), None, p(bws), state, B, H, T, D, dt, scale, lo, hi, p(word), st)
    torch.cuda.synchronize()
    if word is not None:
        assert int(word[0]) == guard
    return o, dq, dk, dv


@pytest.mark.parametrize("entry", ["split", "fused"])
@pytest.mark.parametrize("guard", [0, 1])
def test_ragged_takes_any_variant_pair(guard, entry):
    """The C ABI's guarded calls pair any two variants at lengths that are no
    multiple of 128: pairs that the MFMA kernels do not have, against the chosen
    variant alone."""
    T = 77
    q, k, v, g = (x.cuda() for x in _rand((2, 3, T, 64), 41))
    shift = _c_variant(make_variant("asinh", 16, 8.0, T, shift=True, fast_rho=False))
    clamped = _c_variant(make_variant("asinh", 16, 8.0, T, shift=False))
    softmax = _c_variant(make_variant("softmax"))
    for lo, hi in ((shift, clamped), (clamped, shift), (softmax, shift)):
        got = _abi(q, k, v, g, lo, hi, guard, entry)
        want = _abi(q, k, v, g, lo if guard else hi)
        for a, b, name in zip(got, want, ("o", "dq", "dk", "dv")):
            assert rel_l2(a, b) <= 1e-2, name       # bf16 weights and outputs


@pytest.mark.parametrize("T", [77, 333])
def test_ragged_di_in_float32(T):
    """dP - di where both are near 257 and differ by about 0.02, against float64
    with the kernel's own o: float32 sums of 64 products leave about 5e-5 of the
    difference and bf16 ds 2e-3 of it. (di as two bf16 values is off by up to
    0.004, a fifth of it.)"""
    q, k, v, g = (x.cuda().float() for x in _rand((1, 2, T, 64), 43, dtype="f32"))
    v = 0.01 * v
    v[..., 0], v[..., 1] = 256.0, 1.3671875
    g[..., 2:] *= 0.25
    g[..., :2] = 1.0
    leaves = [x.bfloat16().requires_grad_() for x in (q, k, v)]
    g = g.bfloat16()
    o = flash_attention(*leaves, block=T, kind="softmax")
    dq, dk, _ = torch.autograd.grad(o, leaves, g)
    qd, kd, vd, gd = (x.detach().double() for x in (*leaves, g))
    qs = (qd / 8.0).bfloat16().double()
    s = (qs @ kd.transpose(-1, -2)).masked_fill(
        torch.ones(T, T, device=o.device).triu(1) > 0, -float("inf"))
    dp, di = gd @ vd.transpose(-1, -2), (gd * o.detach().double()).sum(-1, keepdim=True)
    ds = torch.softmax(s, -1) * (dp - di)
    assert rel_l2(dq, ds @ kd / 8.0) <= 1.5e-2
    assert rel_l2(dk, ds.transpose(-1, -2) @ qs) <= 1.5e-2


@pytest.mark.parametrize("B,H,T", [(2, 16, 700), (1, 2, 1300), (4, 16, 1300), (8, 16, 2049)])
def test_ragged_dq_is_the_same_in_every_run(B, H, T):
    """Each 256-key block leaves its share of dq in a slot of its own, and the
    finish adds them in order: fewer key blocks than slots (3 of 8, 6 of 128)
    and more (6 and 9 over 4: the later launches add to the slots of the
    first)."""
    q, k, v, g = (x.cuda() for x in _rand((B, H, T, 64), 47))
    leaves = [x.requires_grad_() for x in (q, k, v)]
    o = flash_attention(*leaves, block=T, kind="softmax")
    runs = [torch.autograd.grad(o, leaves, g, retain_graph=True) for _ in range(4)]
    for r in runs[1:]:
        assert all(torch.equal(a, b) for a, b in zip(r, runs[0]))
    ref = [x.detach()[-1:, -2:].double().requires_grad_() for x in leaves]
    s = (ref[0] @ ref[1].transpose(-1, -2) / 8.0).masked_fill(
        torch.ones(T, T, device=o.device).triu(1) > 0, -float("inf"))
    want = torch.autograd.grad(torch.softmax(s, -1) @ ref[2], ref, g[-1:, -2:].double())
    for a, b, name in zip(runs[0], want, ("dq", "dk", "dv")):
        assert rel_l2(a[-1:, -2:], b) <= 1e-2, name     # bf16 weights and outputs


@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("T,j", [(40, 21), (333, 200), (333, 332), (700, 300)])
@pytest.mark.parametrize("kw", [dict(kind="asinh", n=16, c=8.0, shift=False),
                                dict(kind="asinh", n=16, c=8.0, shift=True, fast_rho=False),
                                dict(kind="softmax")], ids=["clamped", "shift", "softmax"])
def test_ragged_non_finite_rows_stay_apart(T, j, kw, value):
    """A row j of q, k, v or dO that is not finite reaches only what sees it,
    also where the bf16 MFMA kernels share its tile or its 256-key block with
    other rows, or read it again in place of rows past the end. The others are
    those of finite inputs, up to bf16 weights rounded at another maximum."""
    q, k, v, g = (x.cuda() for x in _rand((1, 2, T, 64), 53))

    def run(**bad):
        x = dict(q=q, k=k, v=v, g=g)
        for name in bad:
            x[name] = x[name].clone()
            x[name][0, 1, j] = value
        leaves = [x[n].detach().requires_grad_() for n in "qkv"]
        o = flash_attention(*leaves, block=T, **kw)
        return [t.detach()[0] for t in (o, *torch.autograd.grad(o, leaves, x["g"]))]

    want = run()
    rows = torch.arange(T, device="cuda")
    before, after, rest = rows < j, rows > j, rows != j
    # (output, rows that must not change) for each input with the bad row; the
    # outputs o, dq, dk, dv
    cases = dict(q=[(0, rest), (1, rest), (2, after), (3, after)], k=[(0, before), (1, before)],
                 v=[(0, before), (1, before)], g=[(0, rows >= 0), (1, rest), (2, after), (3, after)])
    for name, checks in cases.items():
        got = run(**{name: True})
        for i, keep in checks:
            assert torch.equal(got[i][0], want[i][0]), (name, i)
            if keep.any():
                assert rel_l2(got[i][1][keep], want[i][1][keep]) <= 1e-2, (name, i)
        if name in "vg":        # (a clamped score is finite)
            assert not torch.isfinite(got[dict(v=0, g=1)[name]][1, j]).any()


@pytest.mark.parametrize("tail", [False, True], ids=["in_range", "out_of_range"])
@pytest.mark.parametrize("T", [77, 333, 700])
def test_ragged_forward_entry_points(T, tail):
    """A guarded call at a ragged length through each forward of the C ABI, the
    backward on the workspace that forward was given: the same outputs bit for
    bit from the MFMA kernels (one call, one call without allocation, prepare
    and forward on the two-variant kernels), and the oracle's. Without a
    workspace the generic kernels run the forward."""
    q, k, v, g = _rand((2, 3, T, 64), 59)
    if tail:
        q[:, :, -1] *= 200.0
        k[:, :, -1] *= 200.0
    want, _ = _oracle(q, k, v, g, None, "bf16", kind="asinh", n=16, c=8.0, range_guard=True)
    x = [t.cuda() for t in (q, k, v, g)]
    var = make_variant("asinh", 16, 8.0, T)
    lo = _c_variant(var._replace(shift=False, inv_stat=True, bounded_scores=True))
    hi = _c_variant(var._replace(shift=True, inv_stat=False, fast_rho=False, precise_output=True))
    bound = min(16.0, var.clamp / 2)
    bounds = (bound, min(1e8, 1e37 / (T * (2 * bound + 1) ** 16)))
    guard = 0 if tail else 1
    first = _abi(*x, lo, hi, guard, "fused", bounds)
    _check_all(first, want[:4], "bf16")
    for entry in ("noalloc", "split", "no_workspace"):
        got = _abi(*x, lo, hi, guard, entry, bounds)
        for a, b, name in zip(got, first, ("o", "dq", "dk", "dv")):
            if entry == "no_workspace":
                assert rel_l2(a, b) <= 1e-2, name       # bf16 weights and outputs
            else:
                assert torch.equal(a, b), (entry, name)


def test_ragged_out_of_range_forms_no_row_twice():
    """Out of range the guarded forward's first launch overflows in most rows;
    the second one writes them all, and the first must not form them again one
    by one (60 times the time at T = 1000). The fastest of ten forwards against
    that of the next whole-block length, with room for a busy machine."""
    times = []
    for T in (1000, 1024):
        q, k, v, _ = (x.cuda() for x in _rand((4, 12, T, 64), 61))
        best = math.inf
        for _ in range(10):
            start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            start.record()
            o = flash_attention(20.0 * q, 20.0 * k, v, block=T, kind="asinh", n=16, c=8.0,
                                range_guard=True)
            end.record()
            end.synchronize()
            best = min(best, start.elapsed_time(end))
        assert torch.isfinite(o).all()
        times.append(best)
    assert times[0] <= 8.0 * times[1], times
