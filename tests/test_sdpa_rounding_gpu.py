"""What the rounding of the probabilities to 16 bits may do to a result. All values of a head are the same row v, so the exact result
is v whatever the scores are, and one key outweighs all others by 2^x with a probability that loses half a unit when it is rounded
relative to the first key, so that the result moves by one unit unless the kernel undoes it in one of two ways: the denominator sums
the rounded probabilities, or the row's reference has moved to that key, whose probability is then 1 exactly."""
import math

import pytest
import torch

import brodiffusion_amd as bd
from helpers import TORCH_DT

pytestmark = pytest.mark.gpu


def one_heavy_key(dtype, d, H, Lq, Lk, at, x, **kw):
    td = TORCH_DT[dtype]
    unit = 2.0 ** -10 if dtype == "fp16" else 2.0 ** -7          # spacing of the 16-bit values from 1 to 2
    # scores in base-2 exponents: 0 for key 0, floor(x) + log2(1 + 0.97 / 2 units) for key `at`, -30 for the others
    q = torch.zeros(Lq, H, d, dtype=td, device="cuda")
    q[:, :, :2] = 1
    k = torch.zeros(Lk, H, d, dtype=td, device="cuda")
    k[1:, :, 0] = -30
    k[at, :, 0], k[at, :, 1] = x, math.log2(1 + 0.97 / 2 * unit)
    v = (1 + torch.arange(d, device="cuda") % 100 / 128.0).to(td).expand(Lk, H, d)
    out = bd.sdpa_forward(*(t.reshape(-1, H * d) for t in (q, k, v)), H, scale=math.log(2.0), split_scratch=False, **kw).view(Lq, H, d)
    # what is left after either way: the other keys' share, 2^-x, times their rounding, 2^-9 or less, far below half a unit of v
    assert torch.equal(out, v[:1].expand_as(out)), f"{(out != v[:1]).float().mean().item():.3f} of the values moved"


def tiles256(H, Lq):
    return H * ((Lq + 255) // 256) / bd.device_info()["compute_units"]


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d,H,Lq", [(40, 8, 10200), (64, 8, 10200), (72, 16, 4096), (80, 16, 4096), (96, 16, 4096), (96, 8, 8300)])
def test_denominators_of_a_full_gpu_sum_what_multiplies_the_values(dtype, d, H, Lq):
    assert tiles256(H, Lq) >= 1
    one_heavy_key(dtype, d, H, Lq, 400, 100, 7)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d,H,Lq,Lk", [(72, 8, 4096, 231), (80, 8, 4096, 231), (96, 8, 3000, 400), (112, 8, 4096, 231), (128, 8, 4096, 231), (160, 8, 4096, 231), (160, 16, 2304, 700),
                                       (72, 16, 4352, 154), (40, 16, 4352, 154)])
def test_reference_moves_to_terms_above_two_to_the_eighth(dtype, d, H, Lq, Lk):
    """Below one 256-row tile per compute unit, and with few keys (the last two)."""
    assert tiles256(H, Lq) < 1 or Lk <= 192
    one_heavy_key(dtype, d, H, Lq, Lk, 150, 9)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [80, 96, 112])
@pytest.mark.parametrize("H,Lq,Lk", [(8, 4096, 231), (8, 2500, 1030), (16, 2000, 300)])
def test_reference_is_the_maximum_of_the_first_two_tiles(dtype, d, H, Lq, Lk):
    one_heavy_key(dtype, d, H, Lq, Lk, 100, 5)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [40, 64, 72, 80, 96, 112, 128, 160])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("H,Lq,Lk,at", [(16, 1285, 190, 40), (16, 1285, 300, 40), (9, 993, 190, 40), (2, 100, 190, 40), (2, 100, 1500, 63)])
def test_few_rows_reference_is_the_maximum_of_the_first_64_keys(dtype, d, masked, H, Lq, Lk, at):
    one_heavy_key(dtype, d, H, Lq, Lk, at, 5, **({"mask": bd.SdpaMask.causal(Lk)} if masked else {}))


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d", [80, 96, 112])
def test_few_rows_reference_is_the_maximum_of_the_first_128_keys_of_two_wavefronts(dtype, d):
    one_heavy_key(dtype, d, 16, 1285, 300, 70, 5, mask=bd.SdpaMask.causal(300))
