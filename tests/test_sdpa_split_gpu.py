"""Key-axis split of the last round of work groups (mi_sdpa_args.split_scratch): a launch whose query tiles do not
fill the GPU a whole number of times cuts the tiles of the last round into pieces for all compute units and merges
the partial results in FP32. The split result must agree with the unsplit launch to rounding (the probabilities of a part
are rounded against its own reference: at most 2 units in the last place) and with the CPU checker to the usual tolerance
(helpers.TOL)."""
import ctypes as C

import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from brodiffusion_amd import _capi as capi
from helpers import assert_close, randn, to_dev, to_np

pytestmark = pytest.mark.gpu


def max_ulp_diff(a, b):
    unit = 2.0 ** -8 if a.dtype == torch.bfloat16 else 2.0 ** -11
    return (a.float() - b.float()).abs().max().item() / (unit * max(1.0, b.float().abs().max().item()))


def split_bytes(q, k, v, H, **kw):
    """What the library says it needs for this call (0 = it would not split)."""
    a = capi.MiSdpaArgs()
    a.struct_size = C.sizeof(a)
    a.dtype = capi.MI_DTYPE_BF16 if q.dtype == torch.bfloat16 else capi.MI_DTYPE_F16
    a.q, a.k, a.v, a.o = q.data_ptr(), k.data_ptr(), v.data_ptr(), q.data_ptr()
    B = q.shape[0] if q.dim() == 3 else 1
    a.batch, a.num_heads, a.head_dim = B, H, q.shape[-1] // H
    a.q_len, a.kv_len = q.shape[-2], k.shape[-2]
    for key, val in kw.items():
        setattr(a, key, val)
    return int(capi.lib().mi_sdpa_split_scratch_bytes(C.byref(a)))


@pytest.mark.parametrize("dtype,B,H,d,Lq,Lk", [
    ("bf16", 1, 24, 128, 4096, 4096),    # 384 tiles on 256 compute units: the last round is half full, tiles cut in two
    ("bf16", 1, 24, 128, 3328, 3328),    # 312 tiles: a nearly empty last round, many parts per tile
    ("bf16", 2, 16, 72, 4352, 4352),     # head_dim 72, batch 2
    ("fp16", 1, 20, 128, 4500, 2500),    # ragged: last query tile partial, key count not a multiple of 64
])
def test_split_matches_unsplit_and_checker(oracle, dtype, B, H, d, Lq, Lk):
    q = randn(8101, (B, Lq, H * d), dtype)
    k, v = randn(8102, (B, Lk, H * d), dtype), randn(8103, (B, Lk, H * d), dtype)
    dq, dk, dv = to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype)
    need = split_bytes(dq, dk, dv, H)
    assert need > 0, "this shape is expected to qualify for the split"
    plain = bd.sdpa_forward(dq, dk, dv, H, split_scratch=False)
    scratch = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")      # stale NaN patterns must not matter
    split = bd.sdpa_forward(dq, dk, dv, H, split_scratch=scratch)
    assert max_ulp_diff(split, plain) <= 2.0
    # sampled rows against the checker (all heads, rows spread over every query tile and its edges)
    rows = np.unique(np.concatenate([np.arange(0, Lq, 97), np.arange(255, Lq, 256), np.arange(256, Lq, 256), [Lq - 1]])).astype(np.int32)
    for b in range(B):
        ref = oracle.sdpa(q[b], k[b], v[b], H, rows=rows)
        assert_close(ref[rows], to_np(split[b])[rows], dtype, f"split batch {b}")
    # the module's own scratch (default) gives the same bits as a lent one, call after call
    again = bd.sdpa_forward(dq, dk, dv, H)
    assert torch.equal(again, split)
    # one byte short: the library falls back to the unsplit launch
    short = bd.sdpa_forward(dq, dk, dv, H, split_scratch=scratch[: need - 16])
    assert torch.equal(short, plain)


@pytest.mark.parametrize("dtype,H,d,L", [("bf16", 24, 128, 3328), ("fp16", 24, 128, 3328), ("bf16", 16, 72, 4352)])
def test_split_tiles_are_as_close_to_the_exact_result_as_whole_ones(dtype, H, d, L):
    """Against 64 bits, over the query tiles that are cut: the probabilities' rounding and the result's make an error of sqrt(2)
    roundings either way; parts rounded to 16 bits before the merge would make it sqrt(3)."""
    q, k, v = (to_dev(randn(8251 + i, (L, H * d), dtype), dtype) for i in range(3))
    whole, split = bd.sdpa_forward(q, k, v, H, split_scratch=False), bd.sdpa_forward(q, k, v, H)
    tiles = L // 256

    def by_tile(x):
        return x.view(tiles, 256, H, d).permute(2, 0, 1, 3).double()
    cut = (by_tile(whole) != by_tile(split)).flatten(2).any(-1)       # (heads, tiles)
    assert 0 < cut.sum().item() < H * tiles
    errors = torch.zeros(2, dtype=torch.float64, device="cuda")
    for h in cut.any(1).nonzero().flatten().tolist():
        qh, kh, vh = (x[:, h * d:(h + 1) * d].double().contiguous() for x in (q, k, v))
        exact = (torch.softmax(qh @ kh.t().contiguous() * d ** -0.5, dim=-1) @ vh).view(tiles, 256, d)[cut[h]]
        for i, x in enumerate((whole, split)):
            errors[i] += (by_tile(x)[h][cut[h]] - exact).square().sum()
    assert errors[1].sqrt() <= 1.05 * errors[0].sqrt(), errors.sqrt().tolist()


def test_split_then_smaller_call_reuses_scratch(oracle):
    dtype, H, d = "bf16", 24, 128
    big = [to_dev(randn(8200 + i, (4096, H * d), dtype), dtype) for i in range(3)]
    small = [to_dev(randn(8210 + i, (3328, H * d), dtype), dtype) for i in range(3)]
    scratch = torch.empty(max(split_bytes(*big, H), split_bytes(*small, H)), dtype=torch.uint8, device="cuda")
    o_big = bd.sdpa_forward(*big, H, split_scratch=scratch)
    o_small = bd.sdpa_forward(*small, H, split_scratch=scratch)
    assert max_ulp_diff(o_small, bd.sdpa_forward(*small, H, split_scratch=False)) <= 2.0
    assert torch.equal(o_big, bd.sdpa_forward(*big, H, split_scratch=scratch))


def test_split_with_fused_q_rope_and_rotated_k_scratch(oracle):
    """The headline call: RoPE on Q while loading, K rotated into the caller's scratch, then the split launch."""
    dtype, H, d, txt, hp, wp = "bf16", 24, 128, 512, 56, 64
    L = txt + hp * wp
    assert L == 4096
    q, k, v = (to_dev(randn(8300 + i, (L, H * d), dtype), dtype) for i in range(3))
    cos, sin = bd.build_axial_rope_tables(txt, hp, wp, d, (16, 56, 56))
    kr = torch.empty_like(k)
    with_split = bd.sdpa_forward(q, k, v, H, rope_q=(cos, sin), rope_k=(cos, sin), rope_k_scratch=kr)
    without = bd.sdpa_forward(q, k, v, H, rope_q=(cos, sin), rope_k=(cos, sin), rope_k_scratch=kr, split_scratch=False)
    assert max_ulp_diff(with_split, without) <= 2.0


def test_calls_that_do_not_split():
    H, d = 24, 128
    q = torch.zeros(4608, H * d, device="cuda", dtype=torch.bfloat16)
    h = q[:4096]
    assert split_bytes(h, h, h, H) > 0
    assert split_bytes(q, q, q, H) == 0                                               # last round 22/32 full: runs faster unsplit
    assert split_bytes(h, h, h, H, mask_mode=capi.MI_MASK_CAUSAL) == 0                # masked: tiles differ in length
    assert split_bytes(q[:2304], q, q, H) == 0                                        # fewer tiles than compute units
    assert split_bytes(h, h, h, 32) == 0                                              # 512 tiles: two full rounds
    assert split_bytes(h, q[:512], q[:512], H) == 0                                   # 8 key tiles: nothing to gain
    q40 = torch.zeros(2, 4096, 320, device="cuda", dtype=torch.float16)
    assert split_bytes(q40, q40, q40, 8) == 0                                         # head_dim 40 runs on the kernel without split


def test_own_split_scratch_is_per_stream():
    """Two streams run split launches of different problems at the same time with the scratch the Python layer lends by
    itself: each stream has its own (a shared one would be written by both launches at once), and every result equals the
    one computed alone, bit for bit."""
    H, d = 24, 128
    probs = []
    for i, L in enumerate((3328, 4096)):
        q, k, v = (to_dev(randn(8300 + 3 * i + j, (1, L, H * d), "bf16"), "bf16") for j in range(3))
        assert split_bytes(q, k, v, H) > 0
        probs.append((q, k, v, bd.sdpa_forward(q, k, v, H)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[], []]
    for _ in range(4):                      # alternate the submissions so that the launches overlap on the GPU
        for s, (q, k, v, _), o in zip(streams, probs, outs):
            with torch.cuda.stream(s):
                o.append(bd.sdpa_forward(q, k, v, H))
    torch.cuda.synchronize()
    from brodiffusion_amd import ops
    keys = [key for key in ops._split_scratch_cache if key[1] in {s.cuda_stream for s in streams}]
    assert len(keys) == 2 and ops._split_scratch_cache[keys[0]].data_ptr() != ops._split_scratch_cache[keys[1]].data_ptr()
    for (_, _, _, ref), o in zip(probs, outs):
        for got in o:
            assert torch.equal(got, ref)


@pytest.mark.parametrize("dtype,d,Lk", [("bf16", 128, 2497), ("fp16", 72, 2559), ("fp16", 128, 2560)])
def test_parts_around_the_last_key(oracle, dtype, d, Lk):
    """The last part ends inside a key tile (or on its edge); the rows behind the last key and between the rows are poisoned."""
    H, Lq = 17, 4096      # 272 tiles, two of the last round per XCD
    q, k, v = randn(8151, (Lq, H * d), dtype), randn(8152, (Lk, H * d), dtype), randn(8153, (Lk, H * d), dtype)
    k[Lk // 2:] *= 2      # parts with references of their own
    dq = to_dev(q, dtype)
    kb, vb = (torch.full((Lk + 70, H * d + 8), float("nan"), device="cuda", dtype=dq.dtype) for _ in range(2))
    kb[:Lk, :H * d], vb[:Lk, :H * d] = to_dev(k, dtype), to_dev(v, dtype)
    assert split_bytes(dq, kb[:Lk], vb[:Lk], H, head_dim=d, num_heads=H) > 0
    out = bd.sdpa_forward(dq, kb[:Lk, :H * d], vb[:Lk, :H * d], H)
    rows = np.unique(np.concatenate([np.arange(0, Lq, 89), np.arange(Lq - 300, Lq, 13)])).astype(np.int32)
    assert_close(oracle.sdpa(q, k, v, H, rows=rows)[rows], to_np(out)[rows], dtype, f"{Lk} keys")


@pytest.mark.parametrize("dtype,B,H,Hkv,d,Lq,Lk", [
    ("bf16", 1, 20, 5, 128, 4500, 2925),     # 360 tiles, the last key tile of 45 keys
    ("fp16", 2, 17, 17, 72, 2048, 3008),     # batch 2, a mask for each item, whole key tiles
])
@pytest.mark.parametrize("seen", ["padding", "few", "one key", "nothing"])
def test_parts_of_the_tiles_that_a_key_mask_leaves(oracle, dtype, B, H, Hkv, d, Lq, Lk, seen):
    """Parts are shares of the list of tiles with a visible key; where it is short ("few", "one key", "nothing") the first part takes its tile whole.
    Tiles without a visible key are not read: NaN there must not matter."""
    q = randn(8161, (B, Lq, H * d), dtype)
    k, v = randn(8162, (B, Lk, Hkv * d), dtype), randn(8163, (B, Lk, Hkv * d), dtype)
    m = np.zeros((B, Lk), np.float32)
    if seen == "padding":
        m[:, :70] = m[:, 300:] = 1
    elif seen == "few":
        m[:, 130::640] = m[:, Lk - 1] = 1
    elif seen == "one key":
        m[:, Lk // 2] = 1
    if B > 1:
        m[1] = np.random.default_rng(8164).integers(0, 2, Lk)
    rep = lambda x: x.reshape(Lk, Hkv, d).repeat(H // Hkv, axis=1).reshape(Lk, H * d)
    dq, dk, dv, dm = to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), torch.from_numpy(m).cuda()
    for b in range(B):
        for j in range(0, Lk, 64):
            if not m[b, j:j + 64].any():
                dk[b, j:j + 64] = dv[b, j:j + 64] = float("nan")
    need = split_bytes(dq, dk, dv, H, num_kv_heads=Hkv, key_mask=dm.data_ptr(), key_mask_batch_stride=Lk)
    assert need > 0
    split = bd.sdpa_forward(dq, dk, dv, H, num_kv_heads=Hkv, key_mask=dm, split_scratch=torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda"))
    plain = bd.sdpa_forward(dq, dk, dv, H, num_kv_heads=Hkv, key_mask=dm, split_scratch=False)
    assert max_ulp_diff(split, plain) <= 2.0
    rows = np.unique(np.concatenate([np.arange(0, Lq, 197), np.arange(255, Lq, 256)])).astype(np.int32)
    for b in range(B):
        assert_close(oracle.sdpa(q[b], rep(k[b]), rep(v[b]), H, key_mask=m[b], rows=rows)[rows], to_np(split[b])[rows], dtype, f"{seen}, batch {b}")


@pytest.mark.parametrize("dtype,d", [("bf16", 128), ("fp16", 72)])
def test_tiles_that_a_key_mask_leaves_uncut(oracle, dtype, d):
    """Whether a query tile is cut depends on the visible key tiles of its batch item (from 24 of these 40 on); pieces of the last round reach from one
    item into the next, cut or not. A tile that is not cut has the bits of an unsplit launch."""
    B, H, Lq, Lk = 4, 11, 1772, 2500         # 308 query tiles: 7 of a group's last round, 3 of the last group's
    q, k, v = (randn(8171 + i, (B, n, H * d), dtype) for i, n in enumerate((Lq, Lk, Lk)))
    m = np.zeros((B, Lk), np.float32)
    m[0, 5:24 * 64:3] = 1                    # 24 tiles
    m[1, 64:24 * 64] = 1                     # 23
    m[2] = 1
    m[3, Lk - 1] = 1
    dq, dk, dv, dm = to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), torch.from_numpy(m).cuda()
    for b in range(B):
        for j in range(0, Lk, 64):
            if not m[b, j:j + 64].any():
                dk[b, j:j + 64] = dv[b, j:j + 64] = float("nan")
    need = split_bytes(dq, dk, dv, H, key_mask=dm.data_ptr(), key_mask_batch_stride=Lk)
    assert need > 0
    split = bd.sdpa_forward(dq, dk, dv, H, key_mask=dm, split_scratch=torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda"))
    plain = bd.sdpa_forward(dq, dk, dv, H, key_mask=dm, split_scratch=False)
    rows = np.unique(np.concatenate([np.arange(0, Lq, 101), np.arange(255, Lq, 256)])).astype(np.int32)
    for b, cut in enumerate((True, False, True, False)):
        assert max_ulp_diff(split[b], plain[b]) <= 2.0 and torch.equal(split[b], plain[b]) != cut, b
        assert_close(oracle.sdpa(q[b], k[b], v[b], H, key_mask=m[b], rows=rows)[rows], to_np(split[b])[rows], dtype, f"batch {b}")


@pytest.mark.parametrize("dtype,H,Hkv,d,L,split_half", [("bf16", 24, 6, 128, 2700, False), ("fp16", 24, 6, 128, 2816, True), ("bf16", 16, 16, 72, 4400, False)])
def test_key_mask_with_rotated_queries_and_keys(oracle, dtype, H, Hkv, d, L, split_half):
    """A masked block's attention as a program calls it: RoPE on Q as it is loaded (a tile of each part anew), K rotated into a scratch, the padding of
    the prompt hidden, the last round cut."""
    q, k, v = randn(8181, (L, H * d), dtype), randn(8182, (L, Hkv * d), dtype), randn(8183, (L, Hkv * d), dtype)
    angle = np.random.default_rng(8184).uniform(-3, 3, (L, d // 2)).astype(np.float32)
    cos, sin = np.cos(angle), np.sin(angle)
    m = np.ones(L, np.float32)
    m[77:512] = 0
    dq, dk, dv, dm = to_dev(q, dtype), to_dev(k, dtype), to_dev(v, dtype), torch.from_numpy(m).cuda()
    tables, kr = (torch.from_numpy(cos).cuda(), torch.from_numpy(sin).cuda()), torch.empty_like(dk)
    assert split_bytes(dq, dk, dv, H, num_kv_heads=Hkv, key_mask=dm.data_ptr(), key_mask_batch_stride=L) > 0

    def call(**kw):
        return bd.sdpa_forward(dq, dk, dv, H, num_kv_heads=Hkv, key_mask=dm, rope_q=tables, rope_k=tables, rope_k_scratch=kr, rope_split_half=split_half, **kw)
    out = call() if split_half else bd.gqa_attention_masked(dq, dk, dv, *tables, d, H, Hkv, dm, Kr=kr)
    plain = call(split_scratch=False)
    assert max_ulp_diff(out, plain) <= 2.0 and not torch.equal(out, plain)
    qr = oracle.rope_apply(q, cos, sin, H, d, split_half=split_half, round_to_dtype=dtype)
    rep = lambda x: x.reshape(L, Hkv, d).repeat(H // Hkv, axis=1).reshape(L, H * d)
    kx = rep(oracle.rope_apply(k, cos, sin, Hkv, d, split_half=split_half, round_to_dtype=dtype))
    rows = np.unique(np.concatenate([np.arange(0, L, 149), np.arange(255, L, 256)])).astype(np.int32)
    assert_close(oracle.sdpa(qr, kx, rep(v), H, key_mask=m, rows=rows)[rows], to_np(out)[rows], dtype, "rotated, masked, cut")
