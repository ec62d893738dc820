"""Q4_K weights against many activation rows on 256 x 128 tiles (gemm_q4k_wide_kernel): tiles that end inside the weight and the activations, few and
many super-blocks, an odd number of them, K shared and whole, stacks, outputs along either axis, with and without bias, against float64.

The tolerance is that of the other Q4_K kernel (test_gpu_q4k_prefill): f32 accumulators that round once per 16 k here, 16 times a super-block in
place of 8, and one f32 rounding per share."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("stack,m,k,n", [
    ((), 8192, 3072, 1000), ((), 7944, 768, 897), ((), 7937, 1280, 1001), ((), 8130, 512, 1024), ((), 6400, 1024, 1025),
    ((), 2568, 10240, 513), ((), 3000, 8192, 1000), ((2,), 3840, 1536, 1000), ((), 12864, 2304, 130)])
def test_edges(device, oracle, monkeypatch, stack, m, k, n, split):
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", split)
    rng = np.random.default_rng(m + k + n)
    s = stack[0] if stack else 1
    blocks = rng.integers(0, 256, (s * m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(s, m, k)).to("cuda:0")
    x = torch.from_numpy(rng.standard_normal((*stack, n, k)).astype(np.float16)).to("cuda:0")
    bias = torch.from_numpy(rng.standard_normal(m).astype(np.float16)).to("cuda:0")
    t = lambda v: Tensor(tuple(v.shape), DType.F16, device, v.contiguous().view(torch.uint8).reshape(-1))
    weight = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (*stack, m, k), device)
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(s, m, k // 256, 2)).to("cuda:0")
    for to in (True, False):  # contiguous along the weight rows, and along the activations
        got = weight.gemm(t(x), t(bias) if to else None, False, True, to).resolve().storage.view(torch.float16)[: s * m * n]
        got = (got.view(s, n, m) if to else got.view(s, m, n).transpose(1, 2)).double()
        for i in range(s):
            xd = x.view(s, n, k)[i].double()
            want = xd @ w[i].T + (bias.double() if to else 0)
            # what the two terms of a weight may reach before they cancel: 63 * 15 * d and 63 * dmin
            mag = xd.abs().view(n, -1, 256).sum(-1) @ (945 * sb[i, ..., 0] + 63 * sb[i, ..., 1]).T + 2
            err = (got[i] - want).abs()
            assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 256 * 2 + 22 + 16) * mag + 2.0**-25).all(), float((err / mag).max())
