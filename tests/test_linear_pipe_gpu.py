"""The projection GEMM's forms with LDS-DMA operand rings at the sizes where they can go wrong: contractions of fewer stages
than the ring has, exactly as many and one more; one row, one 8-feature piece past a tile; 16-bit and INT8 weights, plain and
GEGLU; three problems of different sizes in one launch. test_every_form_around_its_ring goes through every tile size of the rule and asks
the rule itself that it got there; which tiles the other tests get is up to the rule. Against the CPU checker, one
unit in the last place of the result's magnitude (FP32 accumulation and one rounding, as in tests/test_attn_block_gpu.py)."""
import ctypes as C
import os

import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from brodiffusion_amd import _capi as capi
from brodiffusion_amd import build
from helpers import TORCH_DT, randn, to_dev, to_np

pytestmark = pytest.mark.gpu


def _weight(oracle, seed, n_out, n_in, dtype):
    return oracle.round_to(randn(seed, (n_out, n_in), "fp32") / np.sqrt(n_in), dtype)


def _int8(seed, n_out, n_in):
    rng = np.random.default_rng(seed)
    return rng.integers(-128, 128, (n_out, n_in)).astype(np.int8), (rng.uniform(0.5, 1.5, (n_out, 1)) / (74.0 * np.sqrt(n_in))).astype(np.float32)


def _one_ulp(ref, got, dtype, what):
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    assert np.isfinite(got).all(), what
    assert np.all(np.abs(got - ref) <= unit * np.maximum(np.abs(ref), 2.0 ** -6) * 1.05 + 2e-6), what


def _rows(M):
    return np.unique(np.concatenate([[0, M - 1], np.arange(31, M, 97), [r for t in (64, 128, 256) for r in (t - 1, t, M // t * t - 1, M // t * t) if 0 <= r < M]]))


SHAPES = [(65, 40, 64), (65, 40, 128), (63, 32, 192), (1, 8, 256), (130, 96, 320),          # one to five stages
          (513, 1288, 1280), (2049, 648, 640), (1030, 2248, 2240), (8200, 1032, 128), (4099, 1160, 1152)]


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_pipe_linear_matches_checker(oracle, dtype, M, N, K):
    x, w, b = randn(81 + M, (M, K), dtype), _weight(oracle, 82 + N, N, K, dtype), randn(83 + K, (N,), dtype)
    y = to_np(bd.linear_batched(to_dev(w, dtype), to_dev(b, dtype), to_dev(x, dtype)))
    r = _rows(M)
    _one_ulp(oracle.linear(x[r], w, b), y[r], dtype, f"linear {M}x{N}x{K}")


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", SHAPES[:8])
def test_pipe_linear_int8_matches_checker(oracle, dtype, M, N, K):
    x, b = randn(91 + M, (M, K), dtype), randn(93 + K, (N,), dtype)
    w, s = _int8(92 + N, N, K)
    y = to_np(bd.linear_forward_batched_int8w_fp16(torch.from_numpy(w).cuda(), torch.from_numpy(s).cuda(), to_dev(b, dtype), to_dev(x, dtype)))
    r = _rows(M)
    _one_ulp(oracle.linear(x[r], w.astype(np.float32)) * s.reshape(1, -1) + b, y[r], dtype, f"linear int8 {M}x{N}x{K}")


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("int8", [False, True], ids=["w16", "w8"])
@pytest.mark.parametrize("M,N,K", [(65, 72, 64), (127, 8, 128), (129, 200, 320), (1030, 2568, 640), (770, 5128, 1280)])
def test_pipe_geglu_is_the_linear_layer_and_the_gate(oracle, dtype, int8, M, N, K):
    """Against the checker's linear layer in FP32 followed by y = v gelu(g). Bound: one unit u of the output's magnitude; with
    INT8 weights v and g are rounded to the dtype on both sides, and a sum at a rounding boundary may go either way: another
    u |y| from v and u |g| |v gelu'(g)| <= 1.13 u |v g| from g."""
    import math
    x, b = randn(101 + M, (M, K), dtype), randn(103 + K, (2 * N,), dtype)
    r = _rows(M)
    if int8:
        w, s = _int8(102 + N, 2 * N, K)
        y = bd.fused_linear_geglu_int8w(to_dev(x, dtype), torch.from_numpy(w).cuda(), torch.from_numpy(s).cuda(), to_dev(b, dtype))
        lin = oracle.round_to((oracle.linear(x[r], w.astype(np.float32)) * s.reshape(1, -1) + b).astype(np.float32), dtype)
    else:
        w = _weight(oracle, 102 + N, 2 * N, K, dtype)
        y = bd.fused_linear_geglu(to_dev(x, dtype), to_dev(w, dtype), to_dev(b, dtype))
        lin = oracle.linear(x[r], w, b)
    gate = lin[:, N:].astype(np.float64)
    ref = (lin[:, :N] * gate * 0.5 * (1.0 + np.vectorize(math.erf)(gate / math.sqrt(2.0)))).astype(np.float32)
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    bound = unit * (np.abs(ref) + (np.abs(ref) + 1.13 * np.abs(lin[:, :N] * gate) if int8 else 0.0)) * 1.05 + 2e-6
    assert np.all(np.abs(to_np(y)[r] - ref) <= bound), f"geglu {M}x{N}x{K} int8={int8}"


def test_pipe_three_unequal_problems_in_one_launch(oracle):
    """Q from 300 rows of 320 channels, K and V from 77 rows of 768: tiles of all three problems in one row, different
    contractions. The block equals its parts bit for bit (every form accumulates in the same order)."""
    dtype, L, Lc, C, Cc, H = "fp16", 300, 77, 320, 768, 8
    x, ctx = to_dev(randn(111, (L, C), dtype), dtype), to_dev(randn(112, (Lc, Cc), dtype), dtype)
    wq, wo = (to_dev(_weight(oracle, 113 + i, C, C, dtype), dtype) for i in range(2))
    wk, wv = (to_dev(_weight(oracle, 115 + i, C, Cc, dtype), dtype) for i in range(2))
    out = bd.flash_attention_qkvo_forward(x, ctx, wq, None, wk, None, wv, None, wo, None, None, H, False)
    q, k, v = bd.linear_batched(wq, None, x), bd.linear_batched(wk, None, ctx), bd.linear_batched(wv, None, ctx)
    assert torch.equal(bd.linear_batched(wo, None, bd.flash_attention_forward(q, k, v, None, H, False)), out)


RINGS = [(33, 40, 320), (33, 40, 384), (31, 8, 448), (257, 1096, 320), (257, 1096, 384), (257, 1096, 448), (513, 1288, 192), (513, 1288, 256),
         (513, 1288, 320), (2049, 648, 128), (2049, 648, 192), (2049, 648, 256), (4609, 1160, 192), (4000, 1032, 256), (4000, 1032, 320)]


@pytest.mark.parametrize("int8", [False, True], ids=["w16", "w8"])
@pytest.mark.parametrize("M,N,K", RINGS)
def test_pipe_loading_wavefronts_around_the_ring(oracle, int8, M, N, K):
    (test_pipe_linear_int8_matches_checker if int8 else test_pipe_linear_matches_checker)(oracle, "fp16", M, N, K)


@pytest.mark.parametrize("M,N,K", [(129, 200, 192), (1030, 1288, 256), (1030, 1288, 320), (2049, 1032, 128)])
def test_pipe_geglu_loading_wavefronts(oracle, M, N, K):
    test_pipe_geglu_is_the_linear_layer_and_the_gate(oracle, "bf16", False, M, N, K)


@pytest.mark.parametrize("M,N,K", [(65, 40, 64), (300, 1288, 640), (257, 200, 1280)])
def test_pipe_scales_start_at_any_float(oracle, M, N, K):
    """The scales are read four at a time: rows 1 .. N of a longer scale vector (4-byte alignment), N off every tile width, no bias.
    Same bits as from a vector of their own."""
    x = to_dev(randn(121 + M, (M, K), "fp16"), "fp16")
    w, s = (torch.from_numpy(a).cuda() for a in _int8(122 + N, N, K))
    longer = torch.full((N + 2, 1), float("nan"), device="cuda")
    longer[1:-1] = s
    assert longer[1:-1].data_ptr() % 16 == 4
    assert torch.equal(bd.linear_forward_batched_int8w_fp16(w, longer[1:-1], None, x), bd.linear_forward_batched_int8w_fp16(w, s, None, x))


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(1024, 2240, 2240), (962, 2184, 2240), (2048, 1152, 1152), (2048, 640, 2560), (1985, 616, 2560), (1999, 584, 2624)])
def test_tiles_96_features_wide(oracle, dtype, M, N, K):
    """Around 128 x 96 and 64 x 96 tiles, whole and with a ragged last column and ragged last rows; the row behind stays."""
    x = randn(8600 + M, (M, K), dtype)
    w = _weight(oracle, 8601 + N, N, K, dtype)
    b = oracle.round_to(0.3 * randn(8602, (N,), "fp32"), dtype)
    got = bd.linear_batched(to_dev(w, dtype), to_dev(b, dtype), to_dev(x, dtype))
    rows = _rows(M)
    _one_ulp(oracle.linear(x[rows], w, b), to_np(got)[rows], dtype, "plain")
    out = torch.full((M + 1, N), 7.0, dtype=got.dtype, device="cuda")
    bd.linear_batched(to_dev(w, dtype), to_dev(b, dtype), to_dev(x, dtype), out[:M])
    assert torch.equal(out[:M], got) and (out[M:] == 7).all()


@pytest.mark.parametrize("M,N,K", [(2048, 640, 640), (1985, 616, 640), (2000, 584, 64), (4096, 640, 640), (4037, 600, 704), (8192, 320, 128)])
def test_int8_tiles_96_features_wide(oracle, M, N, K):
    x = randn(8700 + M, (M, K), "fp16")
    w, s = _int8(8701 + N, N, K)
    b = oracle.round_to(0.3 * randn(8702, (N,), "fp32"), "fp16")
    out = torch.full((M + 1, N), 7.0, dtype=torch.float16, device="cuda")
    bd.linear_forward_batched_int8w_fp16(torch.from_numpy(w).cuda(), torch.from_numpy(s).cuda(), to_dev(b, "fp16"), to_dev(x, "fp16"), out[:M])
    rows = _rows(M)
    _one_ulp(oracle.linear(x[rows], w.astype(np.float32) * s, b), to_np(out)[rows], "fp16", "int8")
    assert (out[M:] == 7).all()


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("M,N,K", [(2048, 2560, 640), (1985, 2536, 640), (1024, 5120, 1280)])
def test_geglu_tiles_192_rows(oracle, dtype, M, N, K):
    """192 x 128 GEGLU tiles, whole and ragged, against the checker's layer with exact GELU on FP32 halves."""
    x = randn(8800 + M, (M, K), dtype)
    w = _weight(oracle, 8801 + N, 2 * N, K, dtype)
    b = oracle.round_to(0.3 * randn(8802, (2 * N,), "fp32"), dtype)
    out = torch.full((M + 1, N), 7.0, dtype=to_dev(b, dtype).dtype, device="cuda")
    bd.fused_linear_geglu(to_dev(x, dtype), to_dev(w, dtype), to_dev(b, dtype), out[:M])
    rows = _rows(M)
    _one_ulp(oracle.geglu_exact(oracle.linear(x[rows], w, b)), to_np(out)[rows], dtype, "geglu")
    assert (out[M:] == 7).all()


@pytest.mark.parametrize("M,N,K", [(2048, 2560, 640), (1985, 2536, 640)])
def test_int8_geglu_tiles_192_rows(oracle, M, N, K):
    test_pipe_geglu_is_the_linear_layer_and_the_gate(oracle, "fp16", True, M, N, K)


# INT8, GEGLU, form (its place in the table of its kind in csrc/linear_forms.h; 256 compute units), problems in the launch, and the rows, features
# and contraction of each: one stage fewer than the ring has, as many and one more where the rule takes the form with so few, ragged
# rows and features. Not in it: the 256 x 256 tiles (tests/test_linear_large_gpu.py); fewer stages than the ring for 64 x 96 of 16 bits, 128 x 128 and the
# INT8 GEGLU 256 x 64, which are slower than others there.
FORMS = [
    (0, 0, 0, 1, 35, 40, 320), (0, 0, 0, 1, 34, 40, 384), (0, 0, 0, 1, 33, 40, 448),     # 32 x 32
    (0, 0, 1, 1, 457, 552, 320), (0, 0, 1, 1, 558, 456, 384), (0, 0, 1, 1, 577, 424, 448),     # 64 x 32
    (0, 0, 2, 1, 644, 744, 192), (0, 0, 2, 1, 770, 624, 256), (0, 0, 2, 1, 602, 816, 320),     # 64 x 64
    (0, 0, 3, 3, 5413, 80, 320), (0, 0, 3, 3, 5387, 72, 512), (0, 0, 3, 1, 8272, 80, 1472),     # 64 x 96
    (0, 0, 4, 1, 897, 1096, 128), (0, 0, 4, 1, 1286, 784, 192), (0, 0, 4, 1, 1027, 976, 256),     # 128 x 64, loading wavefronts
    (0, 0, 5, 1, 1684, 2384, 128), (0, 0, 5, 1, 2486, 1552, 192), (0, 0, 5, 1, 2445, 1568, 256),     # 128 x 64
    (0, 0, 6, 1, 1421, 1416, 192), (0, 0, 6, 1, 1622, 1240, 256), (0, 0, 6, 1, 1229, 1672, 320),     # 128 x 96
    (0, 0, 7, 1, 1593, 1832, 448), (0, 0, 7, 3, 1027, 904, 448),     # 128 x 128
    (0, 0, 8, 1, 1227, 1608, 64), (0, 0, 8, 1, 1410, 2024, 128), (0, 0, 8, 1, 1563, 1864, 192),     # 128 x 128, two stages
    (0, 0, 9, 1, 2121, 1928, 192), (0, 0, 9, 1, 1944, 2120, 256), (0, 0, 9, 1, 1926, 2104, 320),     # 192 x 128
    (0, 0, 10, 1, 2576, 2376, 128), (0, 0, 10, 1, 2458, 2448, 192), (0, 0, 10, 1, 2181, 2736, 256),     # 256 x 128
    (1, 0, 0, 1, 33, 40, 320), (1, 0, 0, 1, 33, 40, 384), (1, 0, 0, 1, 33, 40, 448),     # 32 x 32
    (1, 0, 1, 1, 417, 600, 192), (1, 0, 1, 1, 454, 560, 256), (1, 0, 1, 1, 520, 488, 320),     # 64 x 64
    (1, 0, 2, 1, 790, 1224, 256), (1, 0, 2, 1, 1218, 776, 320), (1, 0, 2, 1, 1093, 904, 384),     # 64 x 96
    (1, 0, 3, 1, 1220, 784, 128), (1, 0, 3, 1, 781, 1224, 192), (1, 0, 3, 1, 1222, 1176, 256),     # 128 x 64
    (1, 0, 4, 1, 2455, 1864, 128), (1, 0, 4, 1, 2352, 1952, 192), (1, 0, 4, 1, 1480, 1376, 256),     # 128 x 96
    (1, 0, 5, 1, 1413, 2056, 320), (1, 0, 5, 3, 899, 1000, 320),     # 128 x 128
    (1, 0, 6, 1, 1463, 1360, 64), (1, 0, 6, 1, 1289, 1480, 128), (1, 0, 6, 1, 1237, 1616, 192),     # 128 x 128, two stages
    (0, 1, 0, 1, 67, 72, 128), (0, 1, 0, 1, 72, 72, 192), (0, 1, 0, 1, 66, 72, 256),     # 64 x 64
    (0, 1, 1, 1, 842, 1200, 64), (0, 1, 1, 1, 910, 1104, 128), (0, 1, 1, 1, 789, 1224, 192),     # 128 x 64, two stages
    (0, 1, 2, 1, 898, 1120, 256), (0, 1, 2, 1, 1027, 976, 448),     # 128 x 64
    (0, 1, 3, 1, 1871, 1608, 128), (0, 1, 3, 1, 1857, 1616, 192), (0, 1, 3, 1, 1157, 1672, 256),     # 256 x 64
    (0, 1, 4, 1, 2113, 1928, 64), (0, 1, 4, 1, 2151, 1968, 128), (0, 1, 4, 1, 1880, 2184, 192),     # 192 x 128
    (1, 1, 0, 1, 66, 72, 128), (1, 1, 0, 1, 67, 72, 192), (1, 1, 0, 1, 66, 72, 256),     # 64 x 64
    (1, 1, 1, 1, 778, 1232, 64), (1, 1, 1, 1, 777, 1232, 128), (1, 1, 1, 1, 833, 1168, 192),     # 128 x 64, two stages
    (1, 1, 2, 1, 1604, 1888, 256), (1, 1, 2, 1, 1946, 1560, 448),     # 256 x 64
    (1, 1, 3, 1, 2074, 2448, 128), (1, 1, 3, 1, 2351, 2216, 192), (1, 1, 3, 1, 1985, 2064, 256),     # 192 x 128
]


def _form(problems, int8, geglu):
    if not os.path.exists(build.FORMS_LIB):
        build.build_host()
    mnk = (C.c_int * (3 * len(problems)))(*[v for p in problems for v in p])
    return C.CDLL(build.FORMS_LIB).linear_form(mnk, len(problems), int8, geglu, bd.device_info()["compute_units"])


@pytest.mark.parametrize("int8,geglu,form,n,M,N,K", FORMS)
def test_every_form_around_its_ring(oracle, int8, geglu, form, n, M, N, K):
    """x and y are columns of wider buffers with a poisoned border; bounds as in the tests above."""
    assert _form([(M, N, K)] * n, int8, geglu) == form
    dtype, halves = ("fp16", "bf16")[K // 64 % 2], 2 if geglu else 1
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -11
    args, keep, refs, rows = (capi.MiLinearArgs * n)(), [], [], _rows(M)
    for i in range(n):
        x, b = randn(8900 + M + i, (M, K), dtype), randn(8902 + K + i, (halves * N,), dtype)
        if int8:
            w, s = _int8(8901 + N + i, halves * N, K)
            dw, ds = torch.from_numpy(w).cuda(), torch.from_numpy(s).cuda()
            lin = oracle.linear(x[rows], w.astype(np.float32)) * s.reshape(1, -1) + b
        else:
            w = _weight(oracle, 8901 + N + i, halves * N, K, dtype)
            dw, ds, lin = to_dev(w, dtype), None, oracle.linear(x[rows], w, b)
        if geglu and int8:
            lin = oracle.round_to(lin.astype(np.float32), dtype)
        ref = oracle.geglu_exact(lin) if geglu else lin
        slack = np.abs(ref) + 1.13 * np.abs(lin[:, :N] * lin[:, N:]) if geglu and int8 else 0.0
        refs.append((ref, unit * (np.maximum(np.abs(ref), 2.0 ** -6) + slack) * 1.05 + 2e-6))
        dx = torch.full((M + 1, K + 8), float("nan"), device="cuda", dtype=TORCH_DT[dtype])
        dx[:M, :K] = to_dev(x, dtype)
        dy, db = torch.full((M + 1, N + 8), 7.0, device="cuda", dtype=TORCH_DT[dtype]), to_dev(b, dtype)
        keep.append((dx, dw, ds, db, dy))
        a = args[i]
        a.struct_size, a.dtype = C.sizeof(a), capi.MI_DTYPE_BF16 if dtype == "bf16" else capi.MI_DTYPE_F16
        a.x, a.w, a.bias, a.y, a.w_scales = dx.data_ptr(), dw.data_ptr(), db.data_ptr(), dy.data_ptr(), ds.data_ptr() if int8 else None
        a.rows, a.in_features, a.out_features, a.x_row_stride, a.y_row_stride = M, K, N, K + 8, N + 8
        a.stream = torch.cuda.current_stream().cuda_stream
    lib = capi.lib()
    capi.check(lib.mi_linear_geglu_forward(args) if geglu else lib.mi_linear_forward_n(args, n), "linear")
    for (ref, bound), (*_, dy) in zip(refs, keep):
        assert (dy[M:] == 7).all() and (dy[:, N:] == 7).all()
        got = to_np(dy[:M, :N])[rows]
        assert np.isfinite(got).all() and np.all(np.abs(got - ref) <= bound)
