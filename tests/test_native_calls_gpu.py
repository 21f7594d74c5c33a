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
