"""Attention of head_dim 512 in the kernel for long calls (csrc/sdpa_wide_long.hip), which takes launches that fill the GPU: several
heads, grouped K/V heads, rows of wider buffers, Q rotated on load, masks, the key axis in pieces (some of them without visible keys),
NaN and Inf. Against FP32. Each call is checked to be one that the kernel takes (csrc/sdpa_wide_plan.h)."""
import ctypes as C
import os

import pytest
import torch

import brodiffusion_amd as bd
from brodiffusion_amd import build
from helpers import TOL, TORCH_DT

pytestmark = pytest.mark.gpu
D = 512


def _pieces(batch_heads, q_len, kv_len, causal=False, scratch=True):
    """Into how many pieces the call is cut; it must be one for the kernel."""
    if not os.path.exists(build.FORMS_LIB):
        build.build_host()
    pieces, cu = C.c_int(), bd.device_info()["compute_units"]
    assert C.CDLL(build.FORMS_LIB).wide_plan(batch_heads, q_len, kv_len, int(causal), int(scratch), cu, C.byref(pieces))
    return pieces.value


def _inputs(seed, dtype, B, Lq, Lk, Hq=1, Hkv=1, pad=0):
    """(B, L, H D) each, as columns of buffers `pad` wider whose border is NaN"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for L, H in ((Lq, Hq), (Lk, Hkv), (Lk, Hkv)):
        x = torch.full((B, L + (1 if pad else 0), H * D + pad), float("nan"), device="cuda", dtype=TORCH_DT[dtype])[:, :L, :H * D]
        out.append(x.copy_(torch.randn(B, L, H * D, generator=g, device="cuda")))
    return out


def _reference(q, k, v, Hq, see=None):
    B, Lq, Lk, Hkv = q.shape[0], q.shape[1], k.shape[1], k.shape[2] // D
    heads = lambda x, H: x.float().reshape(B, x.shape[1], H, D).transpose(1, 2)
    kf, vf = (heads(x, Hkv).repeat_interleave(Hq // Hkv, 1) for x in (k, v))
    s = torch.matmul(heads(q, Hq).contiguous(), kf.transpose(2, 3).contiguous()) * D ** -0.5
    if see is not None:
        s = s.masked_fill(~see.expand(s.shape), float("-inf"))
    p = torch.softmax(s, 3)
    if see is not None:
        p = torch.where(see.any(3, keepdim=True), p, torch.zeros_like(p))     # rows without a visible key are zero
    return torch.matmul(p, vf.contiguous()).transpose(1, 2).reshape(B, Lq, Hq * D)


def _close(out, ref, v, dtype):
    # (a mean of values with weights rounded to the type, rounded once itself: below 2 u max |v|, and what FP32 sums add)
    u = 2.0 ** (-8 if dtype == "bf16" else -11)
    ok = torch.isfinite(ref)
    assert torch.equal(ok, torch.isfinite(out))
    d = (out.float() - ref)[ok]
    assert d.abs().max().item() <= 2 * u * v[torch.isfinite(v)].abs().max().float().item() + 1e-4
    assert (d.norm() / ref[ok].norm()).item() <= TOL[dtype][0]


@pytest.mark.parametrize("dtype,B,Hq,Hkv,Lq,Lk,pad", [
    ("fp16", 2, 8, 2, 1500, 700, 24),      # 192 tiles, the last of 92 rows; 28 keys in the last step
    ("bf16", 1, 6, 6, 2000, 3001, 8),      # an odd number of steps, two pieces
    ("bf16", 3, 12, 3, 4095, 130, 0),      # 1152 tiles of five steps, two keys in the last
])
def test_heads_groups_and_strides(dtype, B, Hq, Hkv, Lq, Lk, pad):
    q, k, v = _inputs(9100 + Lq, dtype, B, Lq, Lk, Hq, Hkv, pad)
    _pieces(B * Hq, Lq, Lk)
    out = torch.full((B, Lq + 1, Hq * D + 16), 3.0, device="cuda", dtype=TORCH_DT[dtype])
    bd.sdpa_forward(q, k, v, Hq, num_kv_heads=Hkv, out=out[:, :Lq, :Hq * D])
    assert (out[:, Lq:] == 3).all() and (out[:, :, Hq * D:] == 3).all()
    _close(out[:, :Lq, :Hq * D], _reference(q, k, v, Hq), v, dtype)


@pytest.mark.parametrize("split_half", [False, True], ids=["adjacent", "split_half"])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_q_rotated_on_load(dtype, split_half):
    """Bit for bit the stand-alone rotation followed by plain attention, in one piece and in several."""
    H, L = 2, 3000
    q, k, v = (x[0] for x in _inputs(9200, dtype, 1, L, L, H, H))
    ang = torch.empty(L, D // 2, device="cuda").uniform_(-3, 3, generator=torch.Generator(device="cuda").manual_seed(9201))
    rope = (ang.cos(), ang.sin())
    assert _pieces(H, L, L) > 1
    plain = bd.sdpa_forward(bd.rope_apply(q, *rope, D, H, split_half=split_half), k, v, H)
    assert torch.equal(bd.sdpa_forward(q, k, v, H, rope_q=rope, rope_split_half=split_half), plain)
    q, k, v = (x[0] for x in _inputs(9210, dtype, 1, L, 700, 8, 8))
    assert _pieces(8, L, 700, scratch=False) == 1
    plain = bd.sdpa_forward(bd.rope_apply(q, *rope, D, 8, split_half=split_half), k, v, 8, split_scratch=False)
    assert torch.equal(bd.sdpa_forward(q, k, v, 8, rope_q=rope, rope_split_half=split_half, split_scratch=False), plain)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("kind,value", [("valid", (100, 4096)), ("valid", (0, 2500)), ("valid", (1024, 1025)), ("mask", None)])
def test_masks_over_pieces(dtype, kind, value):
    """Four pieces of 1024 keys: valid lengths that leave some of them or all without a visible key or end in one, a key mask that
    hides whole pieces and every second key."""
    B, L = 2, 4096
    q, k, v = _inputs(9300, dtype, B, L, L)
    assert _pieces(B, L, L) == 4
    key = torch.arange(L, device="cuda")
    if kind == "valid":
        n = torch.tensor(value, dtype=torch.int32, device="cuda")
        kw, see = {"kv_valid_len": n}, key[None] < n[:, None]
    else:
        m = torch.ones(B, L, device="cuda")
        m[0, 1024:3072], m[0, :1024:2] = 0, 0
        m[1, :4000] = 0
        kw, see = {"key_mask": m}, m != 0
    scratch = torch.full((300 << 20,), 0xFF, dtype=torch.uint8, device="cuda")
    out, whole = bd.sdpa_forward(q, k, v, 1, split_scratch=scratch, **kw), bd.sdpa_forward(q, k, v, 1, split_scratch=False, **kw)
    _close(out, _reference(q, k, v, 1, see[:, None, None, :]), v, dtype)
    # the whole comes from the other kernel, whose probabilities are rounded against another reference
    assert (out.float() - whole.float()).abs().max().item() <= 2 * 2.0 ** (-8 if dtype == "bf16" else -11) * max(1.0, whole.float().abs().max().item())


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_masks_in_one_piece(dtype):
    """Causal rows (64 heads, two tiles a compute unit) and a valid length beside a key mask."""
    H, L = 64, 1024
    q, k, v = _inputs(9400, dtype, 1, L, L, H, 8)
    assert _pieces(H, L, L, causal=True) == 1
    pos = torch.arange(L, device="cuda")
    out = bd.sdpa_forward(q, k, v, H, num_kv_heads=8, mask=bd.SdpaMask.causal(0))
    _close(out, _reference(q, k, v, H, (pos[None] <= pos[:, None])[None, None]), v, dtype)
    n = torch.tensor([777], dtype=torch.int32, device="cuda")
    m = (torch.rand(1, L, generator=torch.Generator(device="cuda").manual_seed(9401), device="cuda") > 0.5).float()
    m[:, 64:192] = 0
    assert _pieces(H, L, L) == 1
    out = bd.sdpa_forward(q, k, v, H, num_kv_heads=8, kv_valid_len=n, key_mask=m)
    _close(out, _reference(q, k, v, H, ((pos[None] < n[:, None]) & (m != 0))[:, None, None]), v, dtype)


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("where,value", [("q", float("nan")), ("k", float("nan")), ("v", float("nan")), ("q", float("inf")),
                                         ("k", float("inf")), ("k", float("-inf")), ("v", float("-inf"))])
def test_nan_and_inf(dtype, where, value):
    """What the FP32 softmax makes NaN or infinite is so here, in the same places, and the rest is as without."""
    B, L = 2, 4096
    q, k, v = _inputs(9500, dtype, B, L, L)
    assert _pieces(B, L, L) == 4
    {"q": q, "k": k, "v": v}[where][1, 2077, 9] = value
    ref, out = _reference(q, k, v, 1), bd.sdpa_forward(q, k, v, 1)
    assert torch.isfinite(ref[0]).all() and not torch.isfinite(ref[1]).all()
    assert torch.equal(torch.isnan(ref), torch.isnan(out))
    _close(out, ref, v, dtype)
