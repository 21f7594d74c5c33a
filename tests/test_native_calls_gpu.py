"""The operator calls in native code (host/py_ops.cpp) against the Python code behind them (ops.py)."""
import ctypes
import threading

import pytest
import torch

import brodiffusion_amd as bd
from brodiffusion_amd import _capi as capi, build, ops

pytestmark = pytest.mark.gpu


def rand(*shape, dtype=torch.bfloat16, scale=1.0):
    g = torch.Generator(device="cuda").manual_seed(sum(shape) + len(shape))
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def test_operands_without_columns_raise():
    """Rows of no values, and projections to no features: an error, not a division by the row length."""
    x0, w0, w = rand(3, 0), rand(64, 0), rand(64, 64)
    with pytest.raises(RuntimeError):
        bd.flash_attention_qkvo_forward(x0, None, w0, None, w0, None, w0, None, w, None, None, 1, False)
    with pytest.raises(RuntimeError):
        bd.flash_attention_q_with_kv_cached_forward(x0, rand(5, 64), rand(5, 64), w0, None, w, None, None, 1, False)
    empty = rand(0, 64)
    with pytest.raises(RuntimeError):
        bd.mha_forward(rand(3, 64), empty, empty, empty, rand(64, 0), None, None, None, None, None, 1)


def test_a_launch_leaves_the_interpreter_to_other_threads():
    """Against a library whose add waits for another Python thread (tests/cpp/waiting_library.cpp); nothing is launched."""
    x, y = rand(4, 64), rand(4, 64)
    bd.add_inplace_vec(y, x)          # binds the module
    lend = lambda index, nbytes: ops._own_split_scratch(torch.device("cuda", index), nbytes)   # noqa: E731
    gate = ctypes.CDLL(build.WAITING_LIB)
    opener = threading.Timer(0.2, gate.open_gate)
    ops._native.bind(build.WAITING_LIB, lend)
    try:
        opener.start()
        bd.add_inplace_vec(y, x)
    finally:
        ops._native.bind(capi.LIB_PATH, lend)
        opener.join()


def test_threads_on_one_stream_have_scratch_of_their_own():
    """Launches of two threads may come between each other's on a stream they share, so the partial results of a split launch
    must not be in memory that the other thread's launch uses."""
    H = 24
    problems = [tuple(rand(n, H * 128) for _ in range(3)) for n in (3328, 4096)]
    alone = [bd.sdpa_forward(*p, H) for p in problems]
    torch.cuda.synchronize()
    mine = ops._own_split_scratch(torch.device("cuda", torch.cuda.current_device()), 256)
    results, addresses, start = [[], []], [None, None], threading.Barrier(2)

    def work(i):
        addresses[i] = ops._own_split_scratch(mine.device, 256).data_ptr()
        start.wait()
        for _ in range(6):
            results[i].append(bd.sdpa_forward(*problems[i], H))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert len({mine.data_ptr(), *addresses}) == 3
    for got, ref in zip(results, alone):
        assert len(got) == 6 and all(torch.equal(g, ref) for g in got)


def test_scratch_of_a_captured_call_outlives_its_thread():
    """A split launch captured in a thread that then ends: its replay must not write into memory that somebody else has got since."""
    H, L = 24, 3328
    q, k, v = (rand(L, H * 128) for _ in range(3))
    expected, out = bd.sdpa_forward(q, k, v, H), torch.empty_like(q)
    stream, graph, size = torch.cuda.Stream(), torch.cuda.CUDAGraph(), []

    def work():
        with torch.cuda.stream(stream):
            for _ in range(2):
                bd.sdpa_forward(q, k, v, H, out=out)
            stream.synchronize()
            with torch.cuda.graph(graph, stream=stream):
                bd.sdpa_forward(q, k, v, H, out=out)
            size.append(max(ops._split_scratch_cache[key].numel() for key in ops._split_scratch_cache))
    t = threading.Thread(target=work)
    t.start()
    t.join()
    with torch.cuda.stream(stream):
        others = [torch.full((size[0],), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, expected)
        assert all((x == 0x5A).all() for x in others)


def test_a_declined_call_has_launched_nothing():
    """Arguments that only the last steps of a call use are read before the first: nothing reaches a library that refuses every
    launch (tests/cpp/waiting_library.cpp)."""
    x, w = rand(4, 64), rand(64, 64)
    bd.linear_batched(w, None, x)     # binds the module
    lend = lambda index, nbytes: ops._own_split_scratch(torch.device("cuda", index), nbytes)   # noqa: E731
    ops._native.bind(build.WAITING_LIB, lend)
    try:
        good = (x, w, w, w, w, None, 2, w[0].clone(), w[0].clone(), 1e-5, 1e-15, None, None)
        with pytest.raises(RuntimeError, match="stayed closed"):
            ops._native.sana(*good)
        for i, bad in ((9, "eps"), (10, "eps"), (12, rand(3, 64)), (5, rand(3))):
            assert ops._native.sana(*good[:i], bad, *good[i + 1:]) is None
        good = (x, w, w, w, w, None, None, None, None, None, 1, None, None, None, None, None)
        with pytest.raises(RuntimeError, match="stayed closed"):
            ops._native.mha(*good)
        for i, bad in ((4, rand(64, 8)), (8, rand(3)), (9, torch.ones(4, 4, device="cuda")), (14, rand(4, 8)), (15, rand(3, 64))):
            assert ops._native.mha(*good[:i], bad, *good[i + 1:]) is None
    finally:
        ops._native.bind(capi.LIB_PATH, lend)


# ── every operator both ways ──
class _Watched:
    """The native module, noting which calls it took."""

    def __init__(self, module):
        self.module, self.took = module, []

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.module, name)(*args)
            if r is not None:
                self.took.append(name)
            return r
        return call


class _Absent:
    def __getattr__(self, name):
        return lambda *args: None


def both_ways(call, monkeypatch):
    """(what the native call took, its result or error, the Python code's result or error)"""
    bd.add_inplace_vec(rand(1, 8), rand(1, 8))     # binds the module
    watched, results = _Watched(ops._native), []
    for native in (watched, _Absent()):
        with monkeypatch.context() as m:
            m.setattr(ops, "_native", native)
            try:
                r = call()
                results.append([t.clone() for t in (r if isinstance(r, tuple) else (r,))])
            except Exception as e:   # noqa: BLE001 (the two are compared)
                results.append((type(e), str(e)))
    return watched.took, *results


F16 = torch.float16
N, C, H = 130, 256, 4            # rows, columns, heads of 64
W8 = dict(dtype=torch.int8, device="cuda")


def table(rows, half, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    a = torch.rand(rows, half, generator=g, device="cuda") * 6 - 3
    return a.cos(), a.sin()


def int8(rows, cols):
    g = torch.Generator(device="cuda").manual_seed(rows)
    return torch.randint(-127, 128, (rows, cols), generator=g, **W8), torch.full((rows, 1), 1e-3, device="cuda")


def empty(*shape, dtype=torch.bfloat16):
    return torch.zeros(*shape, dtype=dtype, device="cuda")


VALID = {
    "linear": lambda: bd.linear_batched(rand(C, C), None, rand(N, C)),
    "linear bias, Y, 3-D": lambda: bd.linear_batched(rand(64, C), rand(64), rand(2, N, C), empty(2, N, 64)),
    "linear one row": lambda: bd.linear_batched(rand(64, C), rand(64), rand(C)),
    "linear INT8": lambda: bd.linear_forward_batched_int8w_fp16(*int8(64, C), rand(64, dtype=F16), rand(N, C, dtype=F16)),
    "geglu": lambda: bd.fused_linear_geglu(rand(N, C), rand(2 * C, C), rand(2 * C)),
    "geglu INT8": lambda: bd.fused_linear_geglu_int8w(rand(N, C, dtype=F16), *int8(2 * C, C), rand(2 * C, dtype=F16), empty(N, C, dtype=F16)),
    "add": lambda: bd.add_inplace_vec(rand(N, C), rand(N, C)),
    "rms_norm": lambda: bd.rms_norm_rows(rand(N, C), rand(C), 1e-6),
    "rms_norm of a slice": lambda: bd.rms_norm_rows(rand(N, 2 * C)[:, C:], rand(C), 1e-6, empty(N, C)),
    "rope": lambda: bd.rope_apply(rand(N, C), *table(N, 32), 64, H),
    "rope per head, halves": lambda: bd.rope_apply_perhead(rand(N, C), *table(N * H, 32), 64, H, empty(N, C), True),
    "headnorm": lambda: bd.headnorm_rope(rand(N, C), rand(64), 1e-6, None, None, 64, H),
    "headnorm rope cache": lambda: (lambda c: (bd.headnorm_rope(rand(N, C), rand(64), 1e-6, *table(N, 32), 64, H, empty(N, C), c), c))(empty(50, C)),
    "sdpa": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H),
    "sdpa batch, valid, scale": lambda: bd.sdpa_forward(rand(2, N, C), rand(2, 70, C), rand(2, 70, C), H, scale=0.2, out=empty(2, N, C),
                                                         kv_valid_len=torch.tensor([5, 70], dtype=torch.int32, device="cuda")),
    "sdpa GQA, key mask": lambda: bd.sdpa_forward(rand(N, C), rand(70, 64), rand(70, 64), H, num_kv_heads=1, key_mask=(torch.arange(70, device="cuda") % 3 > 0).float()),
    "sdpa prefix, segments": lambda: bd.sdpa_forward(rand(N, C), rand(N, C), rand(N, C), H, k_prefix=rand(33, C), v_prefix=rand(33, C),
                                                     mask=bd.SdpaMask.block_causal(33, [40, N], [73, 33 + N], [1, 0])),
    "sdpa window": lambda: bd.flash_attention_windowed_forward(rand(N, C), rand(N, C), rand(N, C), None, H, 20),
    "sdpa rope, K scratch": lambda: bd.sdpa_forward(rand(N, C), rand(N, C), rand(N, C), H, rope_q=table(N, 32), rope_k=table(N, 32), rope_k_scratch=empty(N, C)),
    "sdpa split, own scratch": lambda: bd.sdpa_forward(rand(3328, 3072), rand(3328, 3072), rand(3328, 3072), 24),
    "sdpa split, lent scratch": lambda: bd.sdpa_forward(rand(3328, 3072), rand(3328, 3072), rand(3328, 3072), 24,
                                                         split_scratch=torch.empty(1 << 27, dtype=torch.uint8, device="cuda")),
    "sdpa never split": lambda: bd.sdpa_forward(rand(3328, 3072), rand(3328, 3072), rand(3328, 3072), 24, split_scratch=False),
    "joint": lambda: bd.joint_attention(rand(N, C), rand(N, C), rand(N, C), *table(N, 32), 64, H),
    "joint Kr, halves": lambda: (lambda kr: (bd.joint_attention(rand(N, C), rand(N, C), rand(N, C), *table(N, 32), 64, H, Kr=kr, split_half=True), kr))(empty(N, C)),
    "gqa": lambda: bd.gqa_attention_masked(rand(N, C), rand(N, 128), rand(N, 128), *table(N, 32), 64, H, 2, torch.ones(N, device="cuda"), Kr=empty(N, 128)),
    "qkvo self": lambda: bd.flash_attention_qkvo_forward(rand(2, N, C), None, *[rand(C, C), None] * 3, rand(C, C), rand(C), None, H, True),
    "qkvo context, mask": lambda: bd.flash_attention_qkvo_forward(rand(N, C), rand(77, 128), rand(C, C), rand(C), rand(C, 128), rand(C), rand(C, 128), rand(C),
                                                                  rand(64, C), None, torch.ones(77, device="cuda"), H, False, empty(N, 64)),
    "qkvo INT8": lambda: bd.flash_attention_qkvo_int8w_fp16(rand(N, C, dtype=F16), None, *[x for _ in range(4) for x in (*int8(C, C), None)], None, H, False),
    "kv cached": lambda: bd.flash_attention_q_with_kv_cached_forward(rand(2, N, C), rand(2, 77, C), rand(2, 77, C), rand(C, C), None, rand(C, C), rand(C),
                                                                     torch.ones(2, 77, device="cuda"), H, False),
    "mha": lambda: bd.mha_forward(rand(N, C), *[rand(C, C, scale=0.06)] * 4, rand(C), None, rand(C), rand(C), None, H),
    "mha buffers, mask": lambda: bd.mha_forward(rand(N, C), *[rand(C, C, scale=0.06)] * 4, None, None, None, None, torch.ones(N, device="cuda"), H,
                                                *[empty(N, C) for _ in range(3)], None, *[empty(N, C) for _ in range(2)]),
    "linear attention": lambda: bd.linear_attention_relu_forward(rand(2, N, C), rand(2, N, C), rand(2, N, C), H),
    "linear attention state": lambda: (lambda ws: (bd.linear_attention_relu_forward(rand(N, C), rand(N, C), rand(N, C), H, workspace=ws, accumulate_state=True,
                                                                                     scratch=False, form=1), ws))(torch.ones(H * 64 * 65, device="cuda")),
    "sana": lambda: bd.sana_self_attention(rand(N, C), *[rand(C, C, scale=0.06)] * 4, None, H),
    "sana norms, capture": lambda: (lambda st: (bd.sana_self_attention(rand(N, C), *[rand(C, C, scale=0.06)] * 4, rand(C), H, nq=rand(C), nk=rand(C), ref_mode="capture",
                                                                        ref_state=st, out=empty(N, C)), st))(torch.empty(H, 65, 64, device="cuda")),
}


@pytest.mark.parametrize("name", list(VALID))
def test_native_and_python_give_the_same(name, monkeypatch):
    took, native, python = both_ways(VALID[name], monkeypatch)
    assert took, "a valid call is expected to run in native code"
    assert isinstance(native, list) and isinstance(python, list), (native, python)
    assert len(native) == len(python) and all(torch.equal(a, b) for a, b in zip(native, python))


INVALID = {
    "linear columns": lambda: bd.linear_batched(rand(C, C), None, rand(N, 64)),
    "linear dtype": lambda: bd.linear_batched(rand(C, C, dtype=F16), None, rand(N, C)),
    "linear bias length": lambda: bd.linear_batched(rand(C, C), rand(64), rand(N, C)),
    "linear slice of X": lambda: bd.linear_batched(rand(C, C), None, rand(N, 2 * C)[:, :C]),
    "linear Y rows": lambda: bd.linear_batched(rand(C, C), None, rand(N, C), empty(N - 1, C)),
    "linear on the host": lambda: bd.linear_batched(rand(C, C), None, rand(N, C).cpu()),
    "linear scales": lambda: bd.linear_forward_batched_int8w_fp16(int8(64, C)[0], torch.ones(63, device="cuda"), None, rand(N, C, dtype=F16)),
    "linear FP32": lambda: bd.linear_batched(rand(C, C, dtype=torch.float32), None, rand(N, C, dtype=torch.float32)),
    "linear 12 columns": lambda: bd.linear_batched(rand(64, 12), None, rand(N, 12)),
    "geglu odd rows": lambda: bd.fused_linear_geglu(rand(N, C), rand(2 * C - 1, C), None),
    "geglu Y": lambda: bd.fused_linear_geglu(rand(N, C), rand(2 * C, C), None, empty(N, 2 * C)),
    "add shapes": lambda: bd.add_inplace_vec(rand(N, C), rand(N, 64)),
    "add transposed": lambda: bd.add_inplace_vec(rand(C, C).t(), rand(C, C)),
    "rms_norm gain": lambda: bd.rms_norm_rows(rand(N, C), rand(64), 1e-6),
    "rms_norm 3-D": lambda: bd.rms_norm_rows(rand(2, N, C), rand(C), 1e-6),
    "rope tables": lambda: bd.rope_apply(rand(N, C), *table(N - 1, 32), 64, H),
    "rope heads": lambda: bd.rope_apply(rand(N, C), *table(N, 32), 64, 3),
    "rope no head": lambda: bd.rope_apply(rand(N, C), *table(N, 32), -64, -H),
    "headnorm one table": lambda: bd.headnorm_rope(rand(N, C), rand(64), 1e-6, table(N, 32)[0], None, 64, H),
    "headnorm cache rows": lambda: bd.headnorm_rope(rand(N, C), rand(64), 1e-6, None, None, 64, H, cache_out=empty(N + 1, C)),
    "sdpa heads": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), 3),
    "sdpa no heads": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), 0),
    "sdpa V rows": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(69, C), H),
    "sdpa batch": lambda: bd.sdpa_forward(rand(2, N, C), rand(70, C), rand(70, C), H),
    "sdpa out": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, out=empty(N, 64)),
    "sdpa half a prefix": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, k_prefix=rand(3, C)),
    "sdpa prefix columns": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, k_prefix=rand(3, 64), v_prefix=rand(3, 64)),
    "sdpa valid lengths": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, kv_valid_len=torch.ones(2, dtype=torch.int32, device="cuda")),
    "sdpa key mask": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, key_mask=torch.ones(69, device="cuda")),
    "sdpa segments": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, mask=bd.SdpaMask.block_causal(0, [N], [70, 3], [0])),
    "sdpa segments end": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, mask=bd.SdpaMask.block_causal(0, [N - 1], [70], [0])),
    "sdpa rope rows": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, rope_q=table(70, 32)),
    "sdpa scratch without rope": lambda: bd.sdpa_forward(rand(N, C), rand(70, C), rand(70, C), H, rope_k_scratch=empty(70, C)),
    "sdpa head dimension": lambda: bd.sdpa_forward(rand(N, 48), rand(70, 48), rand(70, 48), 1),
    "sdpa operand slices": lambda: bd.sdpa_forward(rand(N, C + 4)[:, :C], rand(70, C), rand(70, C), H),
    "joint shapes": lambda: bd.joint_attention(rand(N, C), rand(70, C), rand(70, C), *table(N, 32), 64, H),
    "joint Kr": lambda: bd.joint_attention(rand(N, C), rand(N, C), rand(N, C), *table(N, 32), 64, H, Kr=empty(N, 64)),
    "joint halves without Kr": lambda: bd.joint_attention(rand(N, C), rand(N, C), rand(N, C), *table(N, 32), 64, H, split_half=True),
    "qkvo heads": lambda: bd.flash_attention_qkvo_forward(rand(N, C), None, *[rand(C, C), None] * 3, rand(C, C), None, None, 3, False),
    "qkvo context columns": lambda: bd.flash_attention_qkvo_forward(rand(N, C), rand(77, 128), *[rand(C, C), None] * 3, rand(C, C), None, None, H, False),
    "qkvo scratch": lambda: bd.flash_attention_qkvo_forward(rand(N, C), None, *[rand(C, C), None] * 3, rand(C, C), None, None, H, False,
                                                            scratch=torch.empty(256, dtype=torch.uint8, device="cuda")),
    "kv cached V": lambda: bd.flash_attention_q_with_kv_cached_forward(rand(N, C), rand(77, C), rand(70, C), rand(C, C), None, rand(C, C), None, None, H, False),
    "mha heads": lambda: bd.mha_forward(rand(N, C), *[rand(C, C)] * 4, None, None, None, None, None, 3),
    "mha widths": lambda: bd.mha_forward(rand(N, C), rand(C, C), rand(64, C), rand(C, C), rand(C, C), None, None, None, None, None, H),
    "mha mask": lambda: bd.mha_forward(rand(N, C), *[rand(C, C)] * 4, None, None, None, None, torch.ones(N - 1, device="cuda"), H),
    "mha buffer": lambda: bd.mha_forward(rand(N, C), *[rand(C, C)] * 4, None, None, None, None, None, H, yc=empty(N, 64)),
    "linear attention shapes": lambda: bd.linear_attention_relu_forward(rand(N, C), rand(70, C), rand(70, C), H),
    "linear attention state": lambda: bd.linear_attention_relu_forward(rand(N, C), rand(N, C), rand(N, C), H, accumulate_state=True),
    "linear attention workspace": lambda: bd.linear_attention_relu_forward(rand(N, C), rand(N, C), rand(N, C), H, workspace=torch.empty(64, device="cuda")),
    "linear attention form": lambda: bd.linear_attention_relu_forward(rand(N, C), rand(N, C), rand(N, C), H, form=9),
    "sana one gain": lambda: bd.sana_self_attention(rand(N, C), *[rand(C, C)] * 4, None, H, nq=rand(C)),
    "sana gain length": lambda: bd.sana_self_attention(rand(N, C), *[rand(C, C)] * 4, None, H, nq=rand(64), nk=rand(64)),
    "sana state": lambda: bd.sana_self_attention(rand(N, C), *[rand(C, C)] * 4, None, H, ref_mode="capture", ref_state=torch.empty(H * 64 * 64, device="cuda")),
    "sana heads": lambda: bd.sana_self_attention(rand(N, C), *[rand(C, C)] * 4, None, 3),
}


@pytest.mark.parametrize("name", list(INVALID))
def test_native_and_python_refuse_the_same(name, monkeypatch):
    _, native, python = both_ways(INVALID[name], monkeypatch)
    assert isinstance(native, tuple) and native == python and issubclass(native[0], RuntimeError), (native, python)
