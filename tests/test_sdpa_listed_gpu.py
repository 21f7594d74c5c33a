"""Key masks and block-causal calls on the 256-row kernel. Key masks: tiles without a visible key are taken out of the walk; masks
that hide whole tiles in any place, all keys, or single keys. Block-causal: query tiles of 256 rows inside a segment, across the
border of two, and behind a causal one, all on the general form."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu


@pytest.fixture
def rows256():
    bd.set_sdpa_kernel_choice(2)
    yield
    bd.set_sdpa_kernel_choice(0)


HIDDEN = {
    "first tiles": [(0, 130)], "middle": [(70, 400)], "last tiles": [(300, 601)], "one tile left": [(0, 256), (320, 601)],
    "every other tile": [(64, 128), (192, 256), (320, 384), (448, 512)], "single keys": [(0, 1), (63, 65), (600, 601)], "one key left": [(0, 333), (334, 601)],
    "two tiles left": [(0, 128), (256, 601)],
}


@pytest.mark.parametrize("d", [72, 128])
@pytest.mark.parametrize("prefix", [0, 70])
@pytest.mark.parametrize("name", list(HIDDEN))
def test_hidden_tiles(oracle, rows256, name, prefix, d):
    dtype, H, Hkv, Lq, Lk = "bf16", 4, 2, 290, 601
    q, k, v = randn(9401, (Lq, H * d), dtype), randn(9402, (Lk, Hkv * d), dtype), randn(9403, (Lk, Hkv * d), dtype)
    m = np.ones(Lk, np.float32)
    for a, b in HIDDEN[name]:
        m[a:b] = 0
    rep = lambda x: np.ascontiguousarray(np.repeat(x.reshape(Lk, Hkv, d), H // Hkv, axis=1).reshape(Lk, H * d))
    ref = oracle.sdpa(q, rep(k), rep(v), H, key_mask=m)
    dev = lambda x: to_dev(np.ascontiguousarray(x), dtype)
    kw = {} if prefix == 0 else dict(k_prefix=dev(k[:prefix]), v_prefix=dev(v[:prefix]))
    out = bd.sdpa_forward(dev(q), dev(k[prefix:]), dev(v[prefix:]), H, num_kv_heads=Hkv, key_mask=torch.from_numpy(m).cuda(), **kw)
    assert_close(ref, to_np(out), dtype, name)


def test_every_key_hidden_and_a_hidden_nan(oracle, rows256):
    dtype, H, d, L = "bf16", 2, 128, 300
    q, k, v = (randn(9411 + i, (L, H * d), dtype) for i in range(3))
    m = np.ones((2, L), np.float32)
    m[0] = 0
    m[1, 64:192] = 0
    dq, dk, dv = (torch.stack([to_dev(x, dtype)] * 2) for x in (q, k, v))
    dv[1, 64:192] = float("nan")
    dk[1, 64:192] = float("nan")
    out = bd.sdpa_forward(dq, dk, dv, H, key_mask=torch.from_numpy(m).cuda())
    assert (out[0] == 0).all()
    assert_close(oracle.sdpa(q, k, v, H, key_mask=m[1]), to_np(out[1]), dtype)


@pytest.mark.parametrize("d", [72, 128])
@pytest.mark.parametrize("prefix", [0, 100])
@pytest.mark.parametrize("ends,causal", [([256, 700, 1300], [1, 0, 0]), ([93, 300, 1300], [1, 0, 0]), ([257, 512, 1300], [0, 1, 0]), ([100, 1300], [0, 0]), ([40, 1300], [0, 1])])
def test_block_causal_tiles(oracle, rows256, ends, causal, prefix, d):
    dtype, H = "bf16", 2
    n = ends[-1]
    q = randn(9421, (n, H * d), dtype)
    k, v = randn(9422, (prefix + n, H * d), dtype), randn(9423, (prefix + n, H * d), dtype)
    rows = np.arange(n)
    seg = np.searchsorted(np.array(ends), rows, side="right")
    hi = np.array([prefix + e for e in ends])[seg]
    hi = np.where(np.array(causal)[seg] == 1, np.minimum(hi, prefix + rows + 1), hi).astype(np.int32)
    ref = oracle.sdpa(q, k, v, H, row_lo=np.zeros(n, np.int32), row_hi=hi)
    dev = lambda x: to_dev(np.ascontiguousarray(x), dtype)
    kw = {} if prefix == 0 else dict(k_prefix=dev(k[:prefix]), v_prefix=dev(v[:prefix]))
    mask = bd.SdpaMask.block_causal(prefix, ends, [prefix + e for e in ends], causal)
    out = bd.sdpa_forward(dev(q), dev(k[prefix:]), dev(v[prefix:]), H, mask=mask, **kw)
    assert_close(ref, to_np(out), dtype, f"{ends} {causal} prefix {prefix}")


@pytest.mark.parametrize("d,H,L", [(128, 3, 1300), (72, 5, 1024)])
def test_key_mask_with_a_valid_length_and_denominators(oracle, rows256, d, H, L):
    """Batch items of different valid lengths (one of them 0), tiles hidden on both sides of it; denominators as an output."""
    dtype, B = "bf16", 3
    q, k, v = (randn(9431 + i, (B, L, H * d), dtype) for i in range(3))
    m = np.ones((B, L), np.float32)
    m[:, 64:200] = 0
    m[2, 640:] = 0
    n = [L, 0, 777]
    lse = torch.full((B, H, L), float("nan"), device="cuda")
    out = bd.sdpa_forward(*(to_dev(x, dtype) for x in (q, k, v)), H, key_mask=torch.from_numpy(m).cuda(),
                          kv_valid_len=torch.tensor(n, dtype=torch.int32, device="cuda"), lse_out=lse)
    for b in range(B):
        m[b, n[b]:] = 0
        assert_close(oracle.sdpa(q[b], k[b], v[b], H, key_mask=m[b]), to_np(out[b]), dtype, f"batch {b}")
        if n[b] == 0:
            assert (out[b] == 0).all() and (lse[b] == float("inf")).all()
            continue
        qh, kh = (torch.from_numpy(x[b]).double().view(L, H, d).transpose(0, 1).contiguous() for x in (q, k))
        s = (qh @ kh.transpose(1, 2).contiguous()) * d ** -0.5
        s[:, :, torch.from_numpy(m[b]) == 0] = float("-inf")
        exact = torch.logsumexp(s, -1) / np.log(2.0)       # base 2
        # raw scores below 2^6 summed from 128 products in 32 bits (2^-17), times 0.18, and a sum of at most L rounded exponentials
        assert (lse[b].double().cpu() - exact).abs().max().item() < 2e-5
