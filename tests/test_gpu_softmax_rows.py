"""Softmax with a row per wavefront (softmax_rows_kernel) against float64, at the row lengths where a lane's share changes.

The tolerance, relative to a value: the rounded difference x - max carries 2^-24 of its size into the exponential, the exponential
is good to two units of the last place, the sum adds 32 values per lane at most and six levels across lanes, the quotient is rounded once."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,n", [("f32", 4), ("f32", 252), ("f32", 256), ("f32", 260), ("f32", 1500), ("f32", 2048),
                                  ("f16", 8), ("f16", 504), ("f16", 512), ("f16", 520), ("f16", 1504), ("f16", 4096)])
def test_against_float64(device, dt, n):
    t, d = (torch.float32, DType.F32) if dt == "f32" else (torch.float16, DType.F16)
    x = torch.randn((203, n), generator=torch.Generator("cuda:0").manual_seed(n), device="cuda:0") * 3
    x[0], x[1, 0], x[2] = 0.0, 60.0, -60000.0  # equal values, one that takes it all, very negative ones
    x[3, : n // 2] = -float("inf")
    x[4], x[5, n - 1], x[6, 0] = -float("inf"), float("nan"), float("inf")
    x[7] = -95.0  # results down to the smallest numbers of either type
    x[7, 0] = 0.0
    x = x.to(t)
    # spelled out: torch's own in float64 gives 0 for values below 1e-38 on long rows
    e = torch.exp(x.double() - x.double().amax(-1, keepdim=True))
    want = e / e.sum(-1, keepdim=True)
    got = Tensor((203, n), d, device, x.clone().view(torch.uint8).reshape(-1)).softmax(1).resolve().storage.view(t)[: x.numel()].view(x.shape).double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isnan(want[4:7]).all()
    size = (x.double() - x.double().amax(-1, keepdim=True)).abs().clamp(max=200)
    rel = 2.0**-24 * (size + 4 + 2 + 32 + 6 + 1) + (2.0**-11 if dt == "f16" else 0)
    tiny = 2.0**-25 if dt == "f16" else 2.0**-149 * 2
    ok = ((got - want).abs() <= rel * want + tiny) | torch.isnan(want)
    assert ok.all(), float(((got - want).abs() / want.clamp(min=1e-38))[~torch.isnan(want)].max())
