"""Attention prologue of the model block on MI355X: projections -> attention inputs.

The reference's block (src/algebraic/model.py:166-174) reshapes the q, k, v
projections to (B, H, T, D), RMS-normalises q and k over D with learned gains
(qk_norm), and rotates them with the position tables (apply_rotary,
algebraic.py:172-179). ``attention_prologue`` does all of it, with the
layout change, in one HIP pass that reads the (B, T, 3 d) output of a fused
QKV projection in place; its backward writes the gradient of that buffer in
one pass. Results are those of the unfused operators, rounding included.
"""

from typing import Optional

import torch

from .. import _native


def attention_prologue(qkv: torch.Tensor, n_heads: int, q_gain: Optional[torch.Tensor],
                       k_gain: Optional[torch.Tensor], cos: Optional[torch.Tensor],
                       sin: Optional[torch.Tensor], eps: float = 1e-5):
    """(q, k, v) in (B, H, T, 64) from a (B, T, 3 H 64) projection output.

    q and k are RMS-normalised over the head dimension with the float32 gains
    (both None: no norm) and rotated by the (T, 32) float32 tables (both
    None: no rotation)."""
    if qkv.ndim != 3 or qkv.shape[-1] % 3 or (qkv.shape[-1] // 3) != n_heads * 64:
        raise ValueError("attention_prologue needs a (B, T, 3 * n_heads * 64) projection")
    if qkv.dtype not in (torch.bfloat16, torch.float32):
        raise ValueError("attention_prologue needs bfloat16 or float32 projections")
    if (q_gain is None) != (k_gain is None) or (cos is None) != (sin is None):
        raise ValueError("gains and tables come in pairs")
    T = qkv.shape[1]
    tabs = [None if t is None else t[:T].to(torch.float32).contiguous() for t in (cos, sin)]
    if tabs[0] is not None and tuple(tabs[0].shape) != (T, 32):
        raise ValueError("rotation tables must be (T, 32)")
    return _native.ops().prologue(qkv, q_gain, k_gain, tabs[0], tabs[1], int(n_heads), float(eps))
