"""Q4_K weights against many activation rows (gemm_q4k_kernel without loading wavefronts: more than one workgroup per compute unit) at
the edges of its tiles, against float64.

The tolerance: products sc * q * x are exact in the MFMA, whose f32 accumulator rounds once per 32 k; per super-block d and dmin are
applied in f32 and the sums of x are held to 2^-22; the result is rounded to f16 once."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [
    (8192, 256, 256),    # one super-block
    (8100, 512, 257),    # the last tiles hold 36 weight rows, one activation row
    (4224, 768, 300), (4160, 1280, 321), (3072, 2304, 1000), (2560, 512, 513), (1090, 1024, 1100), (64, 512, 33000), (20000, 256, 65),
])
def test_edges(device, oracle, m, k, n):
    rng = np.random.default_rng(m + k + n)
    blocks = rng.integers(0, 256, (m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(m, k)).to("cuda:0")
    x = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float16)).to("cuda:0")
    bias = torch.from_numpy(rng.standard_normal(m).astype(np.float16)).to("cuda:0")
    t = lambda v: Tensor(tuple(v.shape), DType.F16, device, v.contiguous().view(torch.uint8).reshape(-1))
    weight = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (m, k), device)
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(m, k // 256, 2)).to("cuda:0")
    for to in (True, False):  # contiguous along the weight rows, and along the activations
        got = weight.gemm(t(x), t(bias) if to else None, False, True, to).resolve().storage.view(torch.float16)[: m * n]
        got = (got.view(n, m) if to else got.view(m, n).T).double()
        xd = x.double()
        want = xd @ w.T + (bias.double() if to else 0)
        # what the two terms of a weight may reach before they cancel: 63 * 15 * d and 63 * dmin
        mag = xd.abs().view(n, -1, 256).sum(-1) @ (945 * sb[..., 0] + 63 * sb[..., 1]).T + 2
        err = (got - want).abs()
        assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 256 * 2 + 14) * mag + 2.0**-25).all(), float((err / mag).max())
