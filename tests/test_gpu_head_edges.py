"""The fused head's backward where its two products are cut into chunks:
dh over the vocabulary, the last dE tiles over the tokens.

References: the CPU oracle, and at the benchmark's size dense float64 math on
the GPU. Tolerances as in test_gpu_qknorm_head.py.
"""

import numpy as np
import pytest
import torch

from _tol import assert_bf16, assert_f32, rel_l2, to_np
from algebraic_amd.kernels import fused_head
from oracle import head as OH
from test_gpu_qknorm_head import _head_inputs, _head_run

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N,d,V", [(1, 64, 513), (31, 128, 1025), (33, 256, 4097),
                                   (40, 264, 2047), (257, 128, 8191), (128, 384, 5074)])
def test_chunked_backward_ragged_k(N, d, V):
    """Vocabularies and token counts that are no multiple of the 32-wide k
    stage (a chunk's last stage partial, or its only one), one to many dh
    chunks, one to three output tiles along the width."""
    h, e, t = _head_inputs(N, d, V, N + V, 0.2)
    for kind, n, c in (("alg_ce", 8, 2.0), ("ce", 16, 16.0)):
        got = _head_run(h, e, t, kind=kind, n=n, c=c, block_n=N)
        (obj, tel), (dh, de) = OH.fused_head(to_np(h), to_np(e), to_np(t), kind=kind, n=n, c=c,
                                             dtype="bf16", g_obj=1.0)
        assert abs(got[0] - obj) <= 2e-4 + 2e-3 * abs(obj)
        np.testing.assert_allclose(got[1], tel, rtol=2e-2, atol=2e-4)
        assert_bf16(got[2], dh, what="dh")
        assert rel_l2(got[3], de) <= 1e-2


@pytest.mark.parametrize("chunk_mib", [0, 830])
def test_chunked_backward_at_benchmark_size(monkeypatch, chunk_mib):
    """N=16384, d=768, V=50304: dh whole, the last dE tiles in chunks; and the
    same as two token chunks of 8192 (830 MiB of dz), where dh is cut as well
    and the second launch adds its chunked dE tiles to the first's."""
    if chunk_mib:
        monkeypatch.setenv("ALGX_HEAD_CHUNK_BYTES", str(chunk_mib << 20))
    N, d, V = 16384, 768, 50304
    gen = torch.Generator(device=DEV).manual_seed(23)
    h = torch.randn((N, d), device=DEV, generator=gen).bfloat16().requires_grad_(True)
    e = (0.02 * torch.randn((V, d), device=DEV, generator=gen)).bfloat16().requires_grad_(True)
    t = torch.randint(0, V, (N,), device=DEV, generator=gen)
    obj, tel = fused_head(h, e, t, kind="ce")
    dh, de = torch.autograd.grad(obj, [h, e])
    with torch.no_grad():
        h64, e64 = h.double(), e.double()
        z = h64 @ e64.T
        lse = torch.logsumexp(z, -1, keepdim=True)
        nll = (lse - z.gather(1, t[:, None]))[:, 0]
        dz = torch.exp(z - lse)
        dz[torch.arange(N, device=DEV), t] -= 1.0
        dz /= N
        assert rel_l2(tel, nll) <= 1e-4
        assert rel_l2(dh, dz @ e64) <= 1e-2
        assert rel_l2(de, dz.T @ h64) <= 1e-2


@pytest.mark.parametrize("N,d,V", [(1, 4, 2), (5, 6, 131), (127, 36, 129), (129, 132, 1021),
                                   (130, 128, 4097), (640, 20, 700)])
def test_float32_head_tile_edges(N, d, V):
    """float32: widths with and without whole 16-byte rows, extents around the
    128-wide tiles and the 16-wide k stage, products cut along k (V = 4097,
    N = 640) and whole."""
    rng = np.random.default_rng(N + d + V)
    h = torch.from_numpy(rng.standard_normal((N, d)).astype(np.float32))
    e = torch.from_numpy((rng.standard_normal((V, d)) * 0.15).astype(np.float32))
    t = torch.from_numpy(rng.integers(0, V, N).astype(np.int64))
    for kind, n, c in (("alg_ce", 8, 2.0), ("ce", 16, 16.0)):
        got = _head_run(h, e, t, kind=kind, n=n, c=c, block_n=N)
        (obj, tel), (dh, de) = OH.fused_head(to_np(h), to_np(e), to_np(t), kind=kind, n=n, c=c,
                                             dtype="f32", g_obj=1.0)
        assert abs(got[0] - obj) <= 1e-5 * abs(obj) + 1e-6
        assert_f32(got[1], tel, what="telemetry")
        assert_f32(got[2], dh, what="dh")
        assert_f32(got[3], de, what="dE")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N", [1, 63, 64, 65, 320])
def test_loss_over_token_blocks(N, dtype):
    """Telemetry and objective around the statistics kernel's 64-token blocks,
    with many chunks per token; a target outside the vocabulary has target
    logit 0 (fused_head.py:80)."""
    V, d = 3001, 64
    h, e, t = _head_inputs(N, d, V, 3 + N, 0.2)
    h = h if dtype == "bf16" else h.float()
    t[0] = -1
    t[N // 2] = V + 2
    z = to_np(h) @ to_np(e.bfloat16() if dtype == "bf16" else e).T
    lse = np.log(np.exp(z - z.max(-1, keepdims=True)).sum(-1)) + z.max(-1)
    inside = (t.numpy() >= 0) & (t.numpy() < V)
    zt = np.where(inside, z[np.arange(N), np.where(inside, t.numpy(), 0)], 0.0)
    obj, tel = fused_head(h.to(DEV), e.to(DEV), t.to(DEV), kind="ce", block_n=N)
    # float32 sums of 3001 terms: 1e-6 relative, and one rounding of lse - zt
    np.testing.assert_allclose(to_np(tel), lse - zt, rtol=1e-5, atol=1e-5)
    np.testing.assert_allclose(float(obj), (lse - zt).mean(), rtol=1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["ce", "alg_ce"])
@pytest.mark.parametrize("bad", ["nan", "minus_inf"])
def test_non_finite_target_logit_reaches_the_objective(dtype, kind, bad):
    """A target logit that is NaN (a NaN hidden state) or -inf gives NaN for the
    token and for the objective, so that a trainer stops on it, as the formula
    on materialised logits does; the other tokens keep their values."""
    N, d, V, row = 70, 64, 513, 66
    h, e, t = _head_inputs(N, d, V, 11, 0.2)
    h, e, t = h.to(DEV, dtype), e.to(DEV, dtype), t.to(DEV)
    e[:, 0] = 1.0
    e[t[row], 0] = -1.0
    kw = dict(kind=kind, n=8, c=2.0, block_n=N)
    _, want = fused_head(h, e, t, **kw)
    if bad == "nan":
        h[row] = float("nan")
    else:
        h[row, 0] = float("inf")
    obj, tel = fused_head(h, e, t, **kw)
    others = torch.arange(N, device=DEV) != row
    assert torch.equal(tel[others], want[others])
    assert torch.isnan(tel[row]) and torch.isnan(obj)
