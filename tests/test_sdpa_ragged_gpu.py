"""Calls in which every query row sees the same keys, whatever their number: a length that is no multiple of the 64-key tile,
a valid length per batch item, a cached prefix whose last tile is partial. On the 256-row kernels they run the form that
treats only the last tile of a segment specially; here it meets the edges of tiles (and nothing at all, valid length 0); calls with a key mask on
both sides of the rule that chooses between 128-row and 256-row tiles."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu
DIMS = [("fp16", 40), ("bf16", 64), ("bf16", 72), ("bf16", 128)]


@pytest.mark.parametrize("choice", [0, 2])
@pytest.mark.parametrize("dtype,d", DIMS)
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (33, 63), (257, 65), (64, 127), (300, 129), (256, 191), (31, 577)])
def test_odd_key_counts(oracle, dtype, d, Lq, Lk, choice):
    H = 3
    q, k, v = randn(9301, (Lq, H * d), dtype), randn(9302, (Lk, H * d), dtype), randn(9303, (Lk, H * d), dtype)
    # rows behind the last key are poisoned: reading one would show
    kb, vb = (torch.full((Lk + 70, H * d), float("nan"), device="cuda", dtype=to_dev(q, dtype).dtype) for _ in range(2))
    kb[:Lk], vb[:Lk] = to_dev(k, dtype), to_dev(v, dtype)
    bd.set_sdpa_kernel_choice(choice)
    try:
        out = bd.sdpa_forward(to_dev(q, dtype), kb[:Lk], vb[:Lk], H)
    finally:
        bd.set_sdpa_kernel_choice(0)
    assert_close(oracle.sdpa(q, k, v, H), to_np(out), dtype, f"Lq {Lq} Lk {Lk}")


@pytest.mark.parametrize("dtype,d", DIMS)
def test_valid_lengths_of_a_batch(oracle, dtype, d):
    B, H, Lq, Lk = 6, 2, 70, 330
    valid = [0, 1, 64, 65, 329, 330]
    q, k, v = randn(9311, (B, Lq, H * d), dtype), randn(9312, (B, Lk, H * d), dtype), randn(9313, (B, Lk, H * d), dtype)
    vl = torch.tensor(valid, dtype=torch.int32, device="cuda")
    bd.set_sdpa_kernel_choice(2)
    try:
        out = bd.sdpa_forward(to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), H, kv_valid_len=vl)
    finally:
        bd.set_sdpa_kernel_choice(0)
    assert (out[0] == 0).all()                       # no visible key: a zero row
    for b in range(1, B):
        n = valid[b]
        assert_close(oracle.sdpa(q[b], k[b, :n], v[b, :n], H), to_np(out[b]), dtype, f"valid length {n}")


@pytest.mark.parametrize("dtype,d", [("bf16", 72), ("bf16", 128)])
@pytest.mark.parametrize("Lp,Lk", [(1, 64), (63, 1), (65, 130), (100, 200), (192, 65)])
@pytest.mark.parametrize("wide_rows", [False, True])   # prefix rows of their own stride take the general form
def test_partial_prefix_tiles(oracle, dtype, d, Lp, Lk, wide_rows):
    H, Lq = 2, 200
    q = randn(9321, (Lq, H * d), dtype)
    k, v = randn(9322, (Lp + Lk, H * d), dtype), randn(9323, (Lp + Lk, H * d), dtype)
    def prefix(x):
        t = to_dev(np.ascontiguousarray(x[:Lp]), dtype)
        if not wide_rows:
            return t
        big = torch.full((Lp, 2 * H * d), float("nan"), device="cuda", dtype=t.dtype)
        big[:, :H * d] = t
        return big[:, :H * d]
    bd.set_sdpa_kernel_choice(2)
    try:
        out = bd.sdpa_forward(to_dev(q, dtype), to_dev(np.ascontiguousarray(k[Lp:]), dtype), to_dev(np.ascontiguousarray(v[Lp:]), dtype), H,
                              k_prefix=prefix(k), v_prefix=prefix(v))
    finally:
        bd.set_sdpa_kernel_choice(0)
    assert_close(oracle.sdpa(q, k, v, H), to_np(out), dtype, f"prefix {Lp} + {Lk}")


# Calls of some units of rows per compute unit, on the kernel of their size (few rows, mid sizes) against the forced 128-row kernel
@pytest.mark.parametrize("dtype,d,H,Lq,Lk", [
    ("bf16", 128, 24, 320, 448), ("bf16", 128, 24, 320, 449), ("bf16", 128, 24, 1409, 130), ("bf16", 128, 24, 1409, 128),
    ("bf16", 72, 16, 300, 256), ("bf16", 72, 16, 300, 257), ("fp16", 40, 8, 520, 520), ("fp16", 80, 8, 4096, 1000), ("fp16", 80, 8, 4200, 1000),
])
def test_default_choice_agrees_with_the_128_row_kernel(dtype, d, H, Lq, Lk):
    q, k, v = (to_dev(randn(9331 + i, (n, H * d), dtype), dtype) for i, n in enumerate((Lq, Lk, Lk)))
    got = bd.sdpa_forward(q, k, v, H, split_scratch=False).float()
    bd.set_sdpa_kernel_choice(1)
    try:
        ref = bd.sdpa_forward(q, k, v, H).float()
    finally:
        bd.set_sdpa_kernel_choice(0)
    # both round P (relative 2^-9 / 2^-12 per term) and the result once: a few units of the result's own rounding
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    assert ((got - ref).norm() / ref.norm()).item() <= unit


# (heads, rows, keys): on both sides of the lines between 128-row and 256-row tiles (256 compute units). What turns on them has a mask or
# extras: 12 and 16 key tiles where work groups of 128 rows share compute units and where they do not; at 40 and 64 the 128-row kernel always.
@pytest.mark.parametrize("dtype,d,H,Lq,Lk", [("bf16", 128, 24, 1409, 704), ("bf16", 128, 24, 1409, 705), ("bf16", 128, 24, 320, 960), ("bf16", 128, 24, 320, 961),
                                             ("bf16", 72, 16, 2200, 704), ("bf16", 72, 16, 2200, 705), ("fp16", 40, 8, 3000, 1000), ("bf16", 96, 16, 2100, 1100)])
def test_key_masks_on_both_sides_of_the_256_row_line(oracle, dtype, d, H, Lq, Lk):
    q, k, v = randn(9341, (Lq, H * d), dtype), randn(9342, (Lk, H * d), dtype), randn(9343, (Lk, H * d), dtype)
    shown = np.random.default_rng(Lk).uniform(size=Lk) < 0.8
    out = bd.sdpa_forward(*(to_dev(x, dtype) for x in (q, k, v)), H, key_mask=torch.from_numpy(shown.astype(np.float32)).cuda())
    rows = np.unique(np.concatenate([np.arange(0, Lq, 61), [127, 128, 255, 256, Lq - 1]])).astype(np.int32)
    assert_close(oracle.sdpa(q, np.ascontiguousarray(k[shown]), np.ascontiguousarray(v[shown]), H, rows=rows)[rows], to_np(out)[rows], dtype, f"{shown.sum()} of {Lk} keys")
