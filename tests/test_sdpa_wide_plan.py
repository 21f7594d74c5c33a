"""Which kernel attention of head_dim 512 takes (csrc/sdpa_wide_plan.h): the one for long calls gains by a higher clock at the power
limit, so it takes launches that fill the 256 compute units and no others. The calls are ones timed on both kernels."""
import ctypes as C
import os

import pytest

from brodiffusion_amd import build


@pytest.fixture(scope="module")
def plan():
    if not os.path.exists(build.FORMS_LIB):
        build.build_host()
    lib = C.CDLL(build.FORMS_LIB)

    def ask(batch_heads, q_len, kv_len, causal=False, scratch=True):
        pieces = C.c_int()
        return bool(lib.wide_plan(batch_heads, q_len, kv_len, int(causal), int(scratch), 256, C.byref(pieces))), pieces.value
    return ask


@pytest.mark.parametrize("batch_heads,q_len,kv_len,pieces", [
    (1, 16384, 16384, 2), (1, 9216, 9216, 3), (1, 6400, 6400, 5), (1, 4096, 4096, 6),      # 256, 216, 250 and 192 work groups
    (2, 4096, 4096, 4), (16, 2048, 2048, 1), (48, 600, 600, 1),
    (1024, 128, 128, 1),                                               # 4 key steps a work group
    (640, 128, 1024, 1),                                               # two full rounds and half of one
])
def test_full_gpu_takes_the_kernel_for_long_calls(plan, batch_heads, q_len, kv_len, pieces):
    assert plan(batch_heads, q_len, kv_len) == (True, pieces)


@pytest.mark.parametrize("batch_heads,q_len,kv_len,causal,scratch", [
    (1, 16384, 16384, False, False),      # no scratch for parts: 128 work groups
    (16, 1024, 1024, False, True),        # 128 work groups, not cut
    (10, 2048, 2048, False, False),       # 160
    (18, 2048, 2048, False, False),       # one full round and 32 work groups
    (1, 4096, 4096, True, True), (1, 9216, 9216, True, True), (8, 2048, 2048, True, True), (16, 2048, 2048, True, True),
    (4096, 128, 32, False, True), (2048, 128, 64, False, True),        # 1 and 2 key steps a work group
    (8, 1024, 1024, False, True), (1, 2048, 2048, False, True),        # short
])
def test_other_calls_do_not(plan, batch_heads, q_len, kv_len, causal, scratch):
    assert not plan(batch_heads, q_len, kv_len, causal, scratch)[0]


def test_causal_calls_of_two_tiles_a_compute_unit(plan):
    assert plan(64, 1024, 1024, causal=True) == (True, 1)
