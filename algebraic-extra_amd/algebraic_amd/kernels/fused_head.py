"""Fused tied-embedding projection and likelihood loss on MI355X.

Counterpart of ``algebraic.kernels.fused_head`` (src/algebraic/kernels/fused_head.py):
``fused_head(h, embed, targets, *, kind="ce", n=16, c=16.0, block_n=128,
block_v=512)`` returns ``(objective, telemetry)`` exactly as the reference:

* ``ce``: mean cross-entropy and the per-token NLL ``lse - z_t``;
* ``alg_ce``: likelihood ``p_j ~ rho(z_j/c)^n`` with the argument clamped at
  ``0.25 (1e38/V)^(1/n)``; the objective is ``mean(1 - p_t)`` and its VJP is
  the exact log-likelihood gradient ``(n/c) r_j (p_j - y_j) / N``; the
  telemetry is the target probability.

The (N, V) logits are never materialised: the HIP kernels stream vocabulary
tiles through LDS with bf16 MFMA and keep per-token statistics in registers.
``block_n`` is validated as in the reference (N must be divisible by it);
``block_v`` only documents the caller's tiling.
"""

import math

import torch

from .. import _lib, _native


def _root(value, n):
    out = float(value)
    while n > 1:
        out = math.sqrt(out)
        n //= 2
    return out


def fused_head(h, embed, targets, *, kind="ce", n=16, c=16.0, block_n=128, block_v=512):
    """Fused tied-embedding projection and likelihood objective (fused_head.py:260-275).

    ``h`` (N, d) hidden states, ``embed`` (V, d), ``targets`` (N,). Returns
    ``(objective, telemetry)``; telemetry carries no gradient.
    """
    if kind not in ("ce", "alg_ce"):
        raise ValueError(kind)
    if kind == "alg_ce" and (n & (n - 1)):
        raise ValueError("n must be a power of two")
    N, d = h.shape
    bn = min(block_n, N)
    if N % bn:
        raise ValueError(f"token count {N} must be divisible by block {bn}")
    if h.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("fused_head needs bfloat16 or float32 hidden states")
    if embed.ndim != 2 or embed.shape[1] != d:
        raise ValueError("embed must be (V, d) with the hidden width d")
    clamp = 0.25 * _root(1e38 / embed.shape[0], n) if kind == "alg_ce" else 0.0
    kcode = _lib.HEAD_CE if kind == "ce" else _lib.HEAD_ALG_CE
    return _native.ops().head(h, embed, targets, kcode, int(n), float(c), float(clamp))
