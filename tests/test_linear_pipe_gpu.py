"""The projection GEMM's forms with LDS-DMA operand rings at the sizes where they can go wrong: contractions of fewer stages
than the ring has, exactly as many and one more; one row, one 8-feature piece past a tile; every tile size the dispatch
knows, 16-bit and INT8 weights, plain and GEGLU; three problems of different sizes in one launch. Against the CPU checker, one
unit in the last place of the result's magnitude (FP32 accumulation and one rounding, as in tests/test_attn_block_gpu.py)."""
import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import randn, to_dev, to_np

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


SHAPES = [(65, 40, 64), (65, 40, 128), (63, 32, 192), (1, 8, 256), (130, 96, 320),          # 64 x 32 tiles; 1 to 5 stages, ring of 4
          (513, 1288, 1280), (2049, 648, 640),                                              # 64 x 64, 128 x 64
          (1030, 2248, 2240), (8200, 1032, 128), (4099, 1160, 1152)]                        # 128 x 128 twice, 256 x 128


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


RINGS = [(33, 40, 320), (33, 40, 384), (31, 8, 448),               # 32 x 32 tiles, ring of 6: one stage fewer, as many, one more
         (257, 1096, 320), (257, 1096, 384), (257, 1096, 448),      # 64 x 32, 6
         (513, 1288, 192), (513, 1288, 256), (513, 1288, 320),      # 64 x 64, 4
         (2049, 648, 128), (2049, 648, 192), (2049, 648, 256),      # 128 x 64, 3
         (4609, 1160, 192), (4000, 1032, 256), (4000, 1032, 320)]   # 192 x 128, 4 (its own wavefronts load)


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
    """128 x 96 and 64 x 96 tiles, whole and with a last column of 72, 40 and 8 features and ragged last rows; the row behind stays."""
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
