"""Calls with few query rows: work groups of R x S wavefronts, R groups of 32 rows (1 up to one such unit per compute unit, 2 up to
two; masked calls 4 up to four), S blocks of 32 keys at a time. Unmasked calls of more units, 16 x 1285 rows here, belong to the kernel of
tests/test_sdpa_flow_gpu.py but for those of many keys at head_dim 64 (test_two_groups_to_a_compute_unit). Key counts around a block and around
one round of S blocks, the last rows, cached prefixes that end inside a block, valid lengths, grouped heads and RoPE on the query,
against the CPU checker; infinities and NaN next to rows that do not exist."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu
DIMS = [("fp16", 40), ("bf16", 64), ("bf16", 72), ("fp16", 80), ("bf16", 96), ("bf16", 112), ("bf16", 128), ("fp16", 160)]


def sampled(Lq):
    return np.unique(np.concatenate([np.arange(0, Lq, max(1, Lq // 40)), [min(31, Lq - 1), min(32, Lq - 1), Lq - 1]])).astype(np.int32)


# (heads, rows): R = 1 (twice), R = 2, more units than come here, at 256 compute units; keys around one block, one round of S blocks, two rounds
@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("H,Lq", [(2, 1), (3, 65), (9, 993), (16, 1285)])
@pytest.mark.parametrize("Lk", [1, 32, 33, 129, 257, 515])
def test_rows_and_keys(oracle, dtype, d, H, Lq, Lk):
    q, k, v = randn(9601, (Lq, H * d), dtype), randn(9602, (Lk, H * d), dtype), randn(9603, (Lk, H * d), dtype)
    k[:16] *= 4          # the first block decides most rows: the maxima of the partial results are far apart
    out = bd.sdpa_forward(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), H)
    rows = sampled(Lq)
    assert_close(oracle.sdpa(q, k, v, H, rows=rows)[rows], to_np(out)[rows], dtype, f"{H} x {Lq} rows, {Lk} keys")


@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("H,Lq", [(3, 40), (9, 993), (16, 1285)])
@pytest.mark.parametrize("Lp,Lk", [(1, 64), (31, 1), (33, 130), (64, 33), (300, 95)])
def test_prefix_and_valid_length(oracle, dtype, d, H, Lq, Lp, Lk):
    check_prefix_and_valid_length(oracle, dtype, d, H, Lq, Lp, Lk, (None, 0, 1, Lp, Lp + 1, Lp + Lk - 1))


def check_prefix_and_valid_length(oracle, dtype, d, H, Lq, Lp, Lk, lengths):
    """Prefix rows of a stride of their own; rows behind both segments poisoned."""
    q, k, v = randn(9621, (Lq, H * d), dtype), randn(9622, (Lp + Lk, H * d), dtype), randn(9623, (Lp + Lk, H * d), dtype)
    def placed(x, width):
        t = torch.full((len(x) + 40, width), float("nan"), device="cuda", dtype=to_dev(x[:1], dtype).dtype)
        t[:len(x), :H * d] = to_dev(np.ascontiguousarray(x), dtype)
        return t[:len(x), :H * d]
    kp, vp, kf, vf = placed(k[:Lp], 2 * H * d), placed(v[:Lp], H * d + 8), placed(k[Lp:], H * d), placed(v[Lp:], H * d + 8)
    rows = sampled(Lq)
    dq = to_dev(q, dtype)
    for valid in lengths:
        vl = None if valid is None else torch.tensor([valid], dtype=torch.int32, device="cuda")
        out = bd.sdpa_forward(dq, kf, vf, H, kv_valid_len=vl, **({"k_prefix": kp, "v_prefix": vp} if Lp else {}))
        n = Lp + Lk if valid is None else valid
        if n == 0:
            assert (out == 0).all()
        else:
            assert_close(oracle.sdpa(q, k[:n], v[:n], H, rows=rows)[rows], to_np(out)[rows], dtype, f"prefix {Lp} + {Lk}, valid {valid}")


# head_dim 64, 528 to 1024 units and 48 or more blocks of keys: R = 2 with two groups to a compute unit
@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("H,Lq,Lp,Lk", [(16, 1050, 0, 1505), (8, 4090, 45, 1500), (11, 2000, 1601, 33)])
def test_two_groups_to_a_compute_unit(oracle, dtype, H, Lq, Lp, Lk):
    assert 2 < H * ((Lq + 31) // 32) / bd.device_info()["compute_units"] <= 4 and (Lp + 31) // 32 + (Lk + 31) // 32 >= 48
    v_of = (None, 0, Lp + 1, Lp + Lk - 1) if Lp else (None, 0, 1, 1000, Lk - 1)
    check_prefix_and_valid_length(oracle, dtype, 64, H, Lq, Lp, Lk, v_of)


@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("H,n", [(2, 70), (9, 993), (16, 1285)])
def test_masks(oracle, dtype, d, H, n):
    """Causal rows (whole, and a window whose first blocks are skipped) and block-causal rows behind a cached prefix."""
    Lp = 45
    q = randn(9651, (n, H * d), dtype)
    k, v = randn(9652, (Lp + n, H * d), dtype), randn(9653, (Lp + n, H * d), dtype)
    dev = lambda x: to_dev(np.ascontiguousarray(x), dtype)
    dq, kp, vp, kf, vf = dev(q), dev(k[:Lp]), dev(v[:Lp]), dev(k[Lp:]), dev(v[Lp:])
    rows, t = sampled(n), n // 3
    pos = Lp + np.arange(n)
    cases = [("causal", bd.SdpaMask.causal(Lp), np.zeros(n), pos + 1),
             ("window", bd.SdpaMask.causal(Lp, 40), np.maximum(0, pos + 1 - 40), pos + 1),
             ("blocks", bd.SdpaMask.block_causal(Lp, [t, n], [Lp + t, Lp + n], [1, 0]), np.zeros(n), np.where(np.arange(n) < t, pos + 1, Lp + n))]
    for name, mask, lo, hi in cases:
        out = bd.sdpa_forward(dq, kf, vf, H, k_prefix=kp, v_prefix=vp, mask=mask)
        ref = oracle.sdpa(q, k, v, H, row_lo=lo.astype(np.int32), row_hi=hi.astype(np.int32), rows=rows)
        assert_close(ref[rows], to_np(out)[rows], dtype, f"{name}, {H} x {n}")


# 776 to 1024 units of 32 rows, the most that come here: one and two wavefronts to a row, windows below, of and above a block
@pytest.mark.parametrize("dtype,d", [("fp16", 80), ("bf16", 96), ("fp16", 112), ("bf16", 128)])
@pytest.mark.parametrize("H,n,windows", [(8, 4032, (1, 31, 256, 1024, 4000)), (110, 250, (5, 32, 100)), (24, 1100, (33, 700))])
def test_windows_at_the_most_rows(oracle, dtype, d, H, n, windows):
    q, k, v = (randn(9661 + i, (n, H * d), dtype) for i in range(3))
    dq, dk, dv = (to_dev(x, dtype) for x in (q, k, v))
    rows, pos = sampled(n), np.arange(n)
    for w in windows:
        out = bd.sdpa_forward(dq, dk, dv, H, mask=bd.SdpaMask.causal(0, w))
        ref = oracle.sdpa(q, k, v, H, row_lo=np.maximum(0, pos + 1 - w).astype(np.int32), row_hi=(pos + 1).astype(np.int32), rows=rows)
        assert_close(ref[rows], to_np(out)[rows], dtype, f"window {w}, {H} x {n}")


@pytest.mark.parametrize("split_half", [False, True])
@pytest.mark.parametrize("dtype,d", DIMS)
def test_grouped_heads_batches_and_rope(oracle, dtype, d, split_half):
    B, H, Hkv, Lq, Lk = 2, 6, 2, 70, 140
    q, k, v = randn(9631, (B, Lq, H * d), dtype), randn(9632, (B, Lk, Hkv * d), dtype), randn(9633, (B, Lk, Hkv * d), dtype)
    ang = np.random.default_rng(d).uniform(-3, 3, (Lq, d // 2)).astype(np.float32)
    cos, sin = np.cos(ang), np.sin(ang)
    tq = [torch.from_numpy(t).cuda() for t in (cos, sin)]
    vl = torch.tensor([Lk, 45], dtype=torch.int32, device="cuda")
    out = bd.sdpa_forward(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), H, num_kv_heads=Hkv, rope_q=tq, rope_split_half=split_half, kv_valid_len=vl)
    for b, n in enumerate((Lk, 45)):
        qr = oracle.rope_apply(q[b], cos, sin, H, d, round_to_dtype=dtype, split_half=split_half)
        kk, vv = (np.repeat(x[b, :n].reshape(n, Hkv, d), H // Hkv, axis=1).reshape(n, H * d) for x in (k, v))
        assert_close(oracle.sdpa(qr, kk, vv, H), to_np(out[b]), dtype, f"batch {b}")


@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("H,Lq", [(2, 40), (9, 993), (16, 1285)])
def test_values_of_the_last_row_do_not_leak(dtype, d, H, Lq):
    """Rows past the last key repeat it in LDS: an infinite value there stays an infinity (0 x Inf would make it NaN), and a NaN key in
    one block makes exactly its head NaN whichever wavefront has it."""
    Lk = 75
    q, k, v = (to_dev(randn(9641 + i, (n, H * d), dtype), dtype) for i, n in enumerate((Lq, Lk, Lk)))
    vi = v.clone()
    vi[Lk - 1, 3] = float("inf")
    out = bd.sdpa_forward(q, k, vi, H)
    assert (out[:, 3] == float("inf")).all() and out[:, :3].isfinite().all() and out[:, 4:].isfinite().all()
    for row in (5, 40, Lk - 1):
        kn = k.clone()
        kn[row, d:2 * d] = float("nan")
        out = bd.sdpa_forward(q, kn, v, H)
        assert out[:, d:2 * d].isnan().all() and not out[:, :d].isnan().any() and not out[:, 2 * d:].isnan().any()
