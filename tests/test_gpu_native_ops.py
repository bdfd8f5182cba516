"""The native autograd functions as autograd functions: argument forms, saved
tensors, unused outputs, transforms and streams. Values are compared with the
same operator's plain call, so equality is exact where no atomics take part."""

import pytest
import torch

from _tol import rel_l2
from algebraic_amd.algebraic import add_rms_norm, glu_packed, rms_norm
from algebraic_amd.kernels import flash_attention, fused_head, qk_rms_norm_pair
from algebraic_amd.kernels.prologue import attention_prologue
from algebraic_amd.layout import heads_to_tokens, project

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _randn(*shape, seed=0, dtype=torch.bfloat16):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(shape, generator=gen, device=DEV).to(dtype)


def _attn(sink, **kw):
    q, k, v = (_randn(2, 3, 128, 64, seed=s).requires_grad_() for s in range(3))
    o = flash_attention(q, k, v, sink, kind="asinh", n=16, c=8.0, range_guard=True, **kw)
    return o, (q, k, v)


@pytest.mark.parametrize("form", ["H", "1H11", "one", "bf16", "double", "strided", "list"])
def test_sink_forms(form):
    """Every form that broadcasts to one logit per head, and the gradient in
    the form's own shape and dtype."""
    vals = [0.25, -0.5, 0.75]
    base = torch.tensor(vals, device=DEV)
    sink = {"H": base, "1H11": base.reshape(1, 3, 1, 1), "one": torch.tensor(0.5, device=DEV),
            "bf16": base.bfloat16(), "double": base.double(),
            "strided": torch.stack([base, base], 1)[:, 0], "list": vals}[form]
    want_sink = base if form != "one" else torch.full((3,), 0.5, device=DEV)
    want_sink = want_sink.clone().requires_grad_()
    ref, _ = _attn(want_sink)
    (dref,) = torch.autograd.grad(ref.float().square().sum(), [want_sink])
    if form == "list":
        assert torch.equal(_attn(sink)[0], ref)
        return
    sink = sink.detach().requires_grad_()
    o, _ = _attn(sink)
    (ds,) = torch.autograd.grad(o.float().square().sum(), [sink])
    assert torch.equal(o, ref) and ds.shape == sink.shape and ds.dtype == sink.dtype
    want = dref.sum() if form == "one" else dref.reshape(sink.shape)
    assert rel_l2(ds, want) <= (1e-2 if form == "bf16" else 1e-5)


def test_saved_tensor_hooks_and_unused_outputs():
    """Saved tensors pass through the default hooks, and an output that the
    objective does not use counts as a zero gradient."""
    packed = []

    def pack(t):
        packed.append(t)
        return t.cpu()

    x, r = (_randn(64, 256, seed=s).requires_grad_() for s in (1, 2))
    g = torch.ones(256, device=DEV, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
        s, y = add_rms_norm(x, r, g)
    grads = torch.autograd.grad(y.float().square().sum(), [x, r, g])
    assert packed
    s2, y2 = add_rms_norm(x, r, g)
    want = torch.autograd.grad(y2.float().square().sum() + 0.0 * s2.float().sum(), [x, r, g])
    assert all(torch.equal(a, b) for a, b in zip(grads, want))
    q, k = (_randn(2, 8, 64, seed=s).requires_grad_() for s in (3, 4))
    gq, gk = (torch.ones(64, device=DEV, requires_grad=True) for _ in range(2))
    yq, yk = qk_rms_norm_pair(q, k, gq, gk, block=8)
    dq, dk, dgk = torch.autograd.grad(yq.float().sum(), [q, k, gk])
    assert dq.abs().sum() > 0 and dk.abs().sum() == 0 and dgk.abs().sum() == 0


def test_transforms_stay_refused():
    """torch.func transforms and forward-mode differentiation raise."""
    gu = _randn(8, 32, dtype=torch.float32)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: glu_packed(t, "alu").sum())(gu)
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda t: rms_norm(t, None))(_randn(4, 8, 32))
    import torch.autograd.forward_ad as fwAD
    with fwAD.dual_level(), pytest.raises(RuntimeError):
        rms_norm(fwAD.make_dual(gu, torch.ones_like(gu)), None)


def test_partial_gradients_of_project():
    """Only the wanted product is formed: x alone, w alone, both."""
    x, w = _randn(64, 64, seed=1), _randn(64, 128, seed=2)
    ref = [t.clone().requires_grad_() for t in (x, w)]
    want = torch.autograd.grad((ref[0].float() @ ref[1].float()).sum(), ref)
    for i in range(2):
        leaves = [x.clone(), w.clone()]
        leaves[i].requires_grad_()
        (got,) = torch.autograd.grad(project(*leaves).float().sum(), [leaves[i]])
        assert rel_l2(got, want[i]) <= 1e-2


def test_strided_inputs_and_a_side_stream():
    """Transposed and sliced inputs, and a forward and backward on a stream of
    the caller's, equal the plain call."""
    q, k, v = (_randn(2, 128, 3, 64, seed=s).transpose(1, 2) for s in range(3))
    plain = flash_attention(*(t.contiguous() for t in (q, k, v)))
    assert torch.equal(flash_attention(q, k, v), plain)
    x = _randn(16, 520, seed=7)[:, 8:]
    assert torch.equal(rms_norm(x, None), rms_norm(x.clone(), None))
    a = _randn(2, 3, 32, 64, seed=8)
    assert torch.equal(heads_to_tokens(a.transpose(1, 2)), a.reshape(2, 3, 2048))
    h, e = _randn(128, 64, seed=9).requires_grad_(), _randn(1000, 64, seed=10).requires_grad_()
    t = torch.randint(0, 1000, (128,), device=DEV)
    want = torch.autograd.grad(fused_head(h, e, t)[0], [h, e])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        got = torch.autograd.grad(fused_head(h, e, t)[0], [h, e])
    torch.cuda.current_stream().wait_stream(side)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    qkv = _randn(2, 32, 384, seed=11)
    y = attention_prologue(qkv, 2, None, None, None, None)
    assert all(torch.equal(y[i], qkv[..., 128 * i:128 * (i + 1)].view(2, 32, 2, 64).transpose(1, 2))
               for i in range(3))
