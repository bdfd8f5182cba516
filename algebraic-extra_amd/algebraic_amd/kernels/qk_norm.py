"""QK RMS normalisation with a learned gain on MI355X.

Counterpart of ``algebraic.kernels.qk_norm`` (src/algebraic/kernels/qk_norm.py):
``qk_rms_norm(x, gain, eps=1e-5, *, block=1024)`` with the same validation,
computing ``rms_norm`` (algebraic.py:76-83) forward and its VJP with single-pass
HBM-bound HIP kernels. ``block`` is validated as in the reference (a row
count multiple aligned to 8) and otherwise only documents the caller's tiling.

``qk_rms_norm_pair(q, k, gain_q, gain_k)`` normalises the attention's q and k
in one launch each way; it returns exactly what two ``qk_rms_norm`` calls
return.
"""

import torch

from .. import _native


def _check(x, gain, eps, block):
    if x.ndim < 2 or x.shape[-1] != 64 or tuple(gain.shape) != (64,):
        raise ValueError("QK RMS kernel needs D=64 and a one-dimensional gain")
    if x.dtype not in (torch.bfloat16, torch.float32) or gain.dtype != torch.float32:
        raise ValueError("QK RMS kernel needs float32/BF16 input and float32 gain")
    if block < 8 or block % 8 or x.numel() // 64 % block:
        raise ValueError("QK RMS row count must be divisible by a block aligned to eight rows")
    if eps <= 0:
        raise ValueError("QK RMS epsilon must be positive")


def qk_rms_norm(x, gain, eps=1e-5, *, block=1024):
    """RMS-normalize D=64 rows with a learned float32 gain (qk_norm.py:62-76)."""
    _check(x, gain, eps, block)
    return _native.ops().qk_norm(x, gain, float(eps))


def qk_rms_norm_pair(q, k, gain_q, gain_k, eps=1e-5, *, block=1024):
    """``(qk_rms_norm(q, gain_q), qk_rms_norm(k, gain_k))`` in one launch each way.

    q and k must have the same shape and dtype (the attention's query and key
    tensors); each is validated as ``qk_rms_norm`` validates its input."""
    _check(q, gain_q, eps, block)
    _check(k, gain_k, eps, block)
    if q.shape != k.shape or q.dtype != k.dtype:
        raise ValueError("QK RMS pair needs q and k of one shape and dtype")
    return _native.ops().qk_norm_pair(q, k, gain_q, gain_k, float(eps))
