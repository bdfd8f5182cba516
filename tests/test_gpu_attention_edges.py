"""Attention at the edges of its kernels' blocks and tiles, against the oracle.

Tolerances as in tests/_tol.py; the sink gradient, a float32 sum over batch
and rows of terms formed from the storage dtype, as in test_gpu_attention.py.
"""

import pytest
import torch

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
