"""The operators' native autograd functions (csrc/torch_ops.cpp).

``ops()`` is the extension module ``_ops.so``, built in-tree beside
``libalgx.so`` by ``algebraic-extra_amd/build.py``. There is no fallback: the
operators raise if it is missing.
"""

import os

OPS_PATH = os.path.join(os.path.dirname(os.path.abspath(__file__)), "_ops.so")

_ops = None


def ops():
    """The extension module, imported once."""
    global _ops
    if _ops is None:
        if not os.path.exists(OPS_PATH):
            raise RuntimeError(f"{OPS_PATH} is missing: build it with "
                               "`python algebraic-extra_amd/build.py`")
        import torch  # noqa: F401  (its libraries must be loaded first)
        from . import _ops as module
        _ops = module
    return _ops
