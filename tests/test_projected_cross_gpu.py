"""Cached cross-attention whose query projection runs inside the attention launch (sdpa_small.hip, project_rows): the block operator
against its three parts called one by one. The projection adds in the same order as the stand-alone one and the keys are shared out the
same way up to 96 of them, so up to there the two agree bit for bit; beyond, and against the checker, to the usual tolerance."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import TORCH_DT, assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu


def _int8(g, n_out, n_in):
    """Uniform bytes have a standard deviation of 74: with these scales outputs stay below 8, where one unit in the last place of fp16 is
    at most 3.9e-3 and the tolerances' absolute bound (5e-3) allows one (with scales up to 2.5e-3 they reached 11: units of 7.8e-3)."""
    w = torch.randint(-127, 128, (n_out, n_in), device="cuda", generator=g, dtype=torch.int32).to(torch.int8)
    return w, (torch.rand(n_out, 1, device="cuda", generator=g) + 0.5) / (74.0 * n_in ** 0.5)


@pytest.mark.parametrize("dtype,B,H,d,Lq,C,keys,w8,bias", [
    ("fp16", 2, 8, 40, 1024, 320, 77, False, False),    # SD 1.5 widths, one work group per compute unit
    ("fp16", 2, 8, 80, 1024, 640, 77, True, False),
    ("bf16", 2, 8, 80, 1024, 640, 77, False, True),
    ("fp16", 1, 8, 80, 1153, 640, 96, True, True),      # one row in the last group; three whole key blocks
    ("bf16", 3, 2, 40, 63, 64, 1, False, True),         # one step of the contraction, one key
    ("fp16", 1, 3, 40, 65, 128, 33, True, False),       # two steps, two key blocks
    ("fp16", 1, 8, 40, 1, 192, 32, False, False),       # a whole round; a single row
    ("bf16", 1, 5, 40, 200, 256, 64, False, False),     # a round and one step
    ("fp16", 2, 40, 80, 100, 448, 95, False, True),     # two rounds and one step
    ("fp16", 1, 8, 80, 1100, 576, 77, True, True),      # three whole rounds
    ("fp16", 1, 8, 40, 640, 320, 97, False, False),     # a second turn of key blocks
    ("fp16", 2, 8, 80, 900, 640, 256, True, False),
])
def test_projected_cross_attention(oracle, dtype, B, H, d, Lq, C, keys, w8, bias):
    T, D = TORCH_DT[dtype], H * d
    g = torch.Generator(device="cuda").manual_seed(Lq + C + keys)
    r = lambda *s, scale=1.0: (torch.randn(*s, device="cuda", generator=g) * scale).to(T)
    x, k, v = r(B, Lq, C), r(B, keys, D), r(B, keys, D)
    bq, bo = (r(D, scale=0.3), r(C, scale=0.1)) if bias else (None, None)
    if w8:
        wq, sq = _int8(g, D, C)
        wo, so = _int8(g, C, D)
        got = bd.flash_attention_q_with_kv_cached_int8w_fp16(x, k, v, wq, sq, bq, wo, so, bo, None, H, False)
        q = bd.linear_forward_batched_int8w_fp16(wq, sq, bq, x.reshape(B * Lq, C)).view(B, Lq, D)
        parts = bd.linear_forward_batched_int8w_fp16(wo, so, bo, bd.sdpa_forward(q, k, v, H).reshape(B * Lq, D)).view(B, Lq, C)
    else:
        wq, wo = r(D, C, scale=C ** -0.5), r(C, D, scale=D ** -0.5)
        got = bd.flash_attention_q_with_kv_cached_forward(x, k, v, wq, bq, wo, bo, None, H, False)
        q = bd.linear_batched(wq, bq, x.reshape(B * Lq, C)).view(B, Lq, D)
        parts = bd.linear_batched(wo, bo, bd.sdpa_forward(q, k, v, H).reshape(B * Lq, D)).view(B, Lq, C)
    if keys <= 96:
        assert torch.equal(got, parts)
    else:
        assert_close(to_np(parts).reshape(B * Lq, C), to_np(got).reshape(B * Lq, C), dtype, "against the parts")
    qn, kn, vn = to_np(q), to_np(k), to_np(v)
    wn = to_np(wo) * (to_np(so) if w8 else 1.0)
    for b in range(B):
        att = oracle.round_to(oracle.sdpa(qn[b], kn[b], vn[b], H), dtype)
        assert_close(oracle.linear(att, wn.astype(np.float32), None if bo is None else to_np(bo)), to_np(got[b]), dtype, f"batch {b}")
    # rows next to the ones asked for stay as they are
    wide = torch.full((B * Lq + 1, C), 5.0, device="cuda", dtype=T)
    scratch = torch.empty(bd.flash_attention_scratch_bytes(B, Lq, keys, D, False), dtype=torch.uint8, device="cuda")
    args = (wq, sq, bq, wo, so, bo) if w8 else (wq, bq, wo, bo)
    f = bd.flash_attention_q_with_kv_cached_int8w_fp16 if w8 else bd.flash_attention_q_with_kv_cached_forward
    again = f(x, k, v, *args, None, H, False, out=wide[:B * Lq].view(B, Lq, C), scratch=scratch)
    assert torch.equal(again, got) and (wide[B * Lq:] == 5).all()
