"""Unmasked calls of more than two units (32 query rows of a head) per compute unit: work groups of 4 wavefronts that share 64-key
tiles. Key counts around a tile and around one pass of the two buffers, the last rows, cached prefixes that end inside a tile, valid
lengths, grouped heads, both RoPE conventions, references that have to move, against the CPU checker; infinities next to rows that do
not exist; the sizes on which the choice of the kernel turns, against the forced 128-row kernel."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu
DIMS = [("fp16", 40), ("bf16", 64), ("bf16", 72), ("fp16", 80), ("bf16", 96), ("bf16", 112), ("bf16", 128), ("fp16", 160)]
H, Lq = 17, 993          # 544 units; the last tile of 128 rows has 97


def sampled(n):
    return np.unique(np.concatenate([np.arange(0, n, 37), [31, 32, 127, 128, n - 1]])).astype(np.int32)


@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("Lk", [1, 63, 64, 65, 128, 129, 200, 448, 513])
def test_key_counts(oracle, dtype, d, Lk):
    q, k, v = randn(9701, (Lq, H * d), dtype), randn(9702, (Lk, H * d), dtype), randn(9703, (Lk, H * d), dtype)
    k[Lk // 2:] *= 3          # later keys outgrow the reference that the first tile sets
    # such rows are close to one value row, |V| up to 4.2 for N(0, 1): one unit of bf16 there is 2^-5 = 0.031, above the absolute
    # bound of 0.02 (helpers.TOL); a quarter of it, 0.008, is not
    v *= 0.25
    kb, vb = (torch.full((Lk + 70, H * d), float("nan"), device="cuda", dtype=to_dev(q[:1], dtype).dtype) for _ in range(2))
    kb[:Lk], vb[:Lk] = to_dev(k, dtype), to_dev(v, dtype)          # rows behind the last key are poisoned
    out = bd.sdpa_forward(to_dev(q, dtype), kb[:Lk], vb[:Lk], H)
    rows = sampled(Lq)
    assert_close(oracle.sdpa(q, k, v, H, rows=rows)[rows], to_np(out)[rows], dtype, f"{Lk} keys")


@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("Lp,Lk", [(1, 64), (63, 1), (65, 130), (128, 33), (300, 95)])
def test_prefix_and_valid_length(oracle, dtype, d, Lp, Lk):
    q = randn(9711, (Lq, H * d), dtype)
    k, v = randn(9712, (Lp + Lk, H * d), dtype), randn(9713, (Lp + Lk, H * d), dtype)
    def placed(x, width):          # rows of a stride of their own, poisoned rows behind them
        t = torch.full((len(x) + 70, width), float("nan"), device="cuda", dtype=to_dev(x[:1], dtype).dtype)
        t[:len(x), :H * d] = to_dev(np.ascontiguousarray(x), dtype)
        return t[:len(x), :H * d]
    kp, vp, kf, vf = placed(k[:Lp], 2 * H * d), placed(v[:Lp], H * d + 8), placed(k[Lp:], H * d), placed(v[Lp:], H * d + 8)
    rows = sampled(Lq)
    dq = to_dev(q, dtype)
    for valid in (None, 0, 1, Lp, Lp + 1, Lp + Lk - 1):
        vl = None if valid is None else torch.tensor([valid], dtype=torch.int32, device="cuda")
        out = bd.sdpa_forward(dq, kf, vf, H, k_prefix=kp, v_prefix=vp, kv_valid_len=vl)
        n = Lp + Lk if valid is None else valid
        if n == 0:
            assert (out == 0).all()
        else:
            assert_close(oracle.sdpa(q, k[:n], v[:n], H, rows=rows)[rows], to_np(out)[rows], dtype, f"prefix {Lp} + {Lk}, valid {valid}")


@pytest.mark.parametrize("split_half", [False, True])
@pytest.mark.parametrize("dtype,d", DIMS)
def test_grouped_heads_batches_and_rope(oracle, dtype, d, split_half):
    B, Hq, Hkv, n, Lk = 2, 6, 2, 1500, 140          # 564 units
    q, k, v = randn(9721, (B, n, Hq * d), dtype), randn(9722, (B, Lk, Hkv * d), dtype), randn(9723, (B, Lk, Hkv * d), dtype)
    ang = np.random.default_rng(d).uniform(-3, 3, (n, d // 2)).astype(np.float32)
    cos, sin = np.cos(ang), np.sin(ang)
    vl = torch.tensor([Lk, 45], dtype=torch.int32, device="cuda")
    out = bd.sdpa_forward(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), Hq, num_kv_heads=Hkv, rope_split_half=split_half,
                          rope_q=[torch.from_numpy(t).cuda() for t in (cos, sin)], kv_valid_len=vl)
    rows = sampled(n)
    for b, m in enumerate((Lk, 45)):
        qr = oracle.rope_apply(q[b], cos, sin, Hq, d, round_to_dtype=dtype, split_half=split_half)
        kk, vv = (np.repeat(x[b, :m].reshape(m, Hkv, d), Hq // Hkv, axis=1).reshape(m, Hq * d) for x in (k, v))
        assert_close(oracle.sdpa(qr, kk, vv, Hq, rows=rows)[rows], to_np(out[b])[rows], dtype, f"batch {b}")


@pytest.mark.parametrize("dtype,d", DIMS)
def test_non_finite_values(dtype, d):
    Lk = 139
    q, k, v = (to_dev(randn(9731 + i, (n, H * d), dtype), dtype) for i, n in enumerate((Lq, Lk, Lk)))
    vi = v.clone()
    vi[Lk - 1, 3] = float("inf")          # rows past the last key repeat it in LDS: 0 x Inf must not show
    out = bd.sdpa_forward(q, k, vi, H)
    assert (out[:, 3] == float("inf")).all() and out[:, :3].isfinite().all() and out[:, 4:].isfinite().all()
    for row in (5, 70, Lk - 1):
        kn = k.clone()
        kn[row, d:2 * d] = float("nan")
        out = bd.sdpa_forward(q, kn, v, H)
        assert out[:, d:2 * d].isnan().all() and not out[:, :d].isnan().any() and not out[:, 2 * d:].isnan().any()


# (heads, rows, keys) on both sides of the lines of the rule (256 compute units)
@pytest.mark.parametrize("dtype,d,H,Lq,Lk", [
    ("fp16", 40, 8, 2048, 300), ("fp16", 40, 8, 2049, 300), ("fp16", 40, 8, 5120, 400), ("fp16", 40, 8, 5121, 400), ("fp16", 40, 8, 8448, 400),
    ("bf16", 64, 8, 3000, 1504), ("bf16", 64, 8, 3000, 1505), ("bf16", 72, 16, 4352, 700), ("bf16", 72, 16, 4864, 700), ("bf16", 72, 16, 4097, 300),
    ("bf16", 128, 24, 1344, 1000), ("bf16", 128, 24, 1345, 1000), ("bf16", 128, 24, 1345, 320), ("bf16", 128, 24, 3000, 900), ("fp16", 160, 8, 2100, 300),
])
def test_agrees_with_the_128_row_kernel(dtype, d, H, Lq, Lk):
    q, k, v = (to_dev(randn(9741 + i, (n, H * d), dtype), dtype) for i, n in enumerate((Lq, Lk, Lk)))
    got = bd.sdpa_forward(q, k, v, H).float()
    bd.set_sdpa_kernel_choice(1)
    try:
        ref = bd.sdpa_forward(q, k, v, H).float()
    finally:
        bd.set_sdpa_kernel_choice(0)
    # both round P (relative 2^-9 / 2^-12 per term) and the result once: a few units of the result's own rounding
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    assert ((got - ref).norm() / ref.norm()).item() <= unit
