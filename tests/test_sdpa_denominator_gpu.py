"""Softmax denominators below one 256-row query tile per compute unit: sums of the FP32 exponentials, whichever kernel takes the
call. The probabilities of all keys but one are chosen to lose half a unit when they are rounded to 16 bits for the product
with V, all in one direction, and the values of those keys are 0: the result is v / (1 + sum of p), which shows whether p was
summed before that rounding or after."""
import math

import numpy as np
import pytest
import torch

import brodiffusion_amd as bd
from helpers import TORCH_DT

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("d,Lq,Lk,form", [
    (40, 300, 128, "plain"), (40, 300, 129, "plain"), (64, 300, 128, "plain"), (64, 300, 129, "plain"),      # 256-row tiles from one key tile on
    (72, 300, 320, "plain"), (72, 300, 321, "plain"), (72, 300, 1030, "causal"),                             # from 5 key tiles, masked from 16
    (72, 300, 130, "plain"), (80, 300, 300, "plain"), (160, 300, 300, "plain"),                              # 128 rows
    (80, 4100, 1030, "plain"), (96, 4100, 1024, "plain"),                                                    # more 128-row tiles than CUs
    (40, 4100, 1030, "rope"), (64, 4100, 1030, "rope"), (72, 4100, 1030, "rope"), (80, 4100, 1030, "rope"), (96, 4100, 1030, "rope"),
])
def test_denominator_is_summed_before_the_rounding(dtype, d, Lq, Lk, form):
    H, td = 8, TORCH_DT[dtype]
    assert H * ((Lq + 255) // 256) < bd.device_info()["compute_units"]
    unit = 2.0 ** -11 if dtype == "fp16" else 2.0 ** -8       # spacing of the 16-bit values from 1/2 to 1
    # scores in base-2 exponents: 0 for key 0, log2(p) for the others, p = 1/2 + 0.97 / 2 units (rounds to 1/2)
    lo = torch.tensor(math.log2(1 + 0.97 * unit)).to(td)
    q = torch.zeros(Lq, H, d, dtype=td, device="cuda")
    q[:, :, :2] = 1
    k = torch.zeros(Lk, H, d, dtype=td, device="cuda")
    k[1:, :, 0], k[1:, :, 1] = -1, lo.item()
    v = torch.zeros(Lk, H, d, dtype=td, device="cuda")
    v0 = (1 + torch.arange(d) / 128.0).to(td)
    v[0] = v0.cuda()
    kw = {}
    if form == "causal":
        kw["mask"] = bd.SdpaMask.causal(Lk)                   # every key visible, on the masked form
    if form == "rope":                                        # K rotated tile by tile, by an angle of 0
        kw["rope_k"] = (torch.ones(Lk, d // 2, device="cuda"), torch.zeros(Lk, d // 2, device="cuda"))
    out = bd.sdpa_forward(*(x.view(-1, H * d) for x in (q, k, v)), H, scale=math.log(2.0), split_scratch=False, **kw)
    p = 2.0 ** (-1 + lo.double().item())
    exact, rounded_first = (v0.double().numpy() / (1 + (Lk - 1) * x) for x in (p, 0.5))
    def to16(x):
        return torch.from_numpy(x).to(td).double().numpy()    # (from 64 bits directly)
    # columns whose exact value is clear of a rounding boundary by more than FP32 sums are off (Lk 2^-24), and that tell the two apart
    clear = (to16(exact * (1 + 2.0 ** -14)) == to16(exact)) & (to16(exact * (1 - 2.0 ** -14)) == to16(exact))
    tell = clear & (to16(exact) != to16(rounded_first))
    assert tell.sum() >= d // 8
    got = out.view(Lq, H, d).double().cpu().numpy()
    assert np.array_equal(got[:, :, tell], np.broadcast_to(to16(exact)[tell], (Lq, H, int(tell.sum()))))
