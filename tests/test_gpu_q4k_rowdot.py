"""One f16 vector against Q4_K weights of K above 4096 (gemv_q4k_rowdot_kernel): steps of 64 vectors per row that end full and ragged, one, two and
four rows per wavefront with the last group short, on both sides of the sizes at which the number of rows changes, stacks, against float64.

The tolerance: every product is exact in f32; a lane adds 32 of them per step, two terms of scales and activation sums, and six additions join the lanes:
2^-24 of what a weight's two terms reach before they cancel for each, and the rounding to f16."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("stacks,m,k", [
    (1, 12289, 4352), (1, 12287, 5376), (1, 6145, 5632), (1, 12289, 5632),   # four rows at three steps (K to 5376), two from four steps on
    (1, 3072, 7424), (1, 3073, 7168), (1, 3073, 7424), (1, 4095, 8960), (1, 4097, 8192), (1, 4096, 10752), (1, 6145, 9216),
    (2, 1537, 8192), (2, 2048, 7424), (1, 1531, 10240)])
def test_against_float64(device, oracle, stacks, m, k):
    rng = np.random.default_rng(m + k)
    blocks = rng.integers(0, 256, (stacks * m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float32).reshape(stacks, m, k)).to("cuda:0").double()
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).reshape(stacks, m, k // 256, 2)).to("cuda:0").double()
    x, bias = rng.standard_normal((stacks, 1, k)).astype(np.float16), rng.standard_normal(m).astype(np.float16)
    shape = (stacks,) if stacks > 1 else ()
    W = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (*shape, m, k), device)
    got = W.gemm(Tensor.from_data(x.reshape(*shape, 1, k), None, device), Tensor.from_data(bias, None, device), False, True, True).resolve().storage
    got = got.view(torch.float16)[: stacks * m].view(stacks, m).double()
    X, b = torch.from_numpy(x).to("cuda:0").double(), torch.from_numpy(bias).to("cuda:0").double()
    want = (w * X).sum(-1) + b
    mag = ((945 * sb[..., 0] + 63 * sb[..., 1]) * X.abs().view(stacks, 1, k // 256, 256).sum(-1)).sum(-1) + b.abs()
    steps = -(-9 * (k // 256) // 64)
    err = (got - want).abs()
    assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (steps * 20 + 8) * mag + 2.0**-25).all(), float((err / mag).max())
