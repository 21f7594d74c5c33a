"""Launches with at most one 128-row query tile per compute unit at head_dim 80, 96 and 112: the wavefronts of a work group take
key blocks in turn and merge. Key counts around the pairs of tiles, rows around the query tile, masks that leave some
of them without keys, a partial prefix, and scores far apart between them."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,d", [("fp16", 80), ("bf16", 96), ("bf16", 112)])
@pytest.mark.parametrize("Lq,Lk", [(1, 193), (64, 256), (65, 257), (130, 320), (31, 385), (200, 511), (64, 449)])
def test_pairs_of_tiles(oracle, dtype, d, Lq, Lk):
    H = 3
    q, k, v = randn(9501, (Lq, H * d), dtype), randn(9502, (Lk, H * d), dtype), randn(9503, (Lk, H * d), dtype)
    k[:64] *= 4          # the first (even) tile decides most rows: the halves' maxima are far apart
    out = bd.sdpa_forward(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), H)
    assert_close(oracle.sdpa(q, k, v, H), to_np(out), dtype, f"Lq {Lq} Lk {Lk}")


@pytest.mark.parametrize("prefix", [0, 100])
def test_causal_rows_and_valid_lengths(oracle, prefix):
    dtype, d, H, n = "fp16", 80, 2, 300
    q = randn(9511, (n, H * d), dtype)
    k, v = randn(9512, (prefix + n, H * d), dtype), randn(9513, (prefix + n, H * d), dtype)
    dev = lambda x: to_dev(np.ascontiguousarray(x), dtype)
    kw = {} if prefix == 0 else dict(k_prefix=dev(k[:prefix]), v_prefix=dev(v[:prefix]))
    out = bd.sdpa_forward(dev(q), dev(k[prefix:]), dev(v[prefix:]), H, mask=bd.SdpaMask.causal(prefix), **kw)
    hi = (prefix + np.arange(n) + 1).astype(np.int32)
    assert_close(oracle.sdpa(q, k, v, H, row_lo=np.zeros(n, np.int32), row_hi=hi), to_np(out), dtype, "causal")
    for valid in (0, 1, 64, 65, 129):
        vl = torch.tensor([valid], dtype=torch.int32, device="cuda")
        out = bd.sdpa_forward(dev(q), dev(k[prefix:]), dev(v[prefix:]), H, kv_valid_len=vl, **kw)
        if valid == 0:
            assert (out == 0).all()
        else:
            assert_close(oracle.sdpa(q, k[:valid], v[:valid], H), to_np(out), dtype, f"valid length {valid}")


def test_a_non_finite_score_stays_visible():
    d, H, n = 80, 2, 256
    q, k, v = (torch.randn(n, H * d, device="cuda", dtype=torch.float16) for _ in range(3))
    for row in (3, 70):                       # in a tile of either half
        kk = k.clone()
        kk[row, :d] = float("nan")
        out = bd.sdpa_forward(q, kk, v, H)
        assert out[:, :d].isnan().all() and not out[:, d:].isnan().any()
