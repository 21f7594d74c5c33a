"""The operator calls in native code (host/py_ops.cpp) against the Python code behind them (ops.py)."""
import pytest
import torch

import brodiffusion_amd as bd

pytestmark = pytest.mark.gpu


def rand(*shape, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + len(shape))
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def test_operands_without_columns_raise():
    """Rows of no values, and projections to no features: an error, not a division by the row length."""
    x0, w0, w = rand(3, 0), rand(64, 0), rand(64, 64)
    with pytest.raises(RuntimeError):
        bd.flash_attention_qkvo_forward(x0, None, w0, None, w0, None, w0, None, w, None, None, 1, False)
    with pytest.raises(RuntimeError):
        bd.flash_attention_q_with_kv_cached_forward(x0, rand(5, 64), rand(5, 64), w0, None, w, None, None, 1, False)
    empty = rand(0, 64)
    with pytest.raises(RuntimeError):
        bd.mha_forward(rand(3, 64), empty, empty, empty, rand(64, 0), None, None, None, None, None, 1)
