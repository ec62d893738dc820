"""Q4_K weights against many activation rows on 256 x 128 tiles (gemm_q4k_wide_kernel): tiles that end inside the weight and the activations, one, few and
many super-blocks, an odd number of them, K shared and whole, stacks, outputs along either axis, bias along either, activations on both ways of
storing, against float64.  Each size is one that the launcher's estimate gives this kernel: SHARED with a workspace, WHOLE with one and without.

The tolerance is that of the other Q4_K kernel (test_gpu_q4k_prefill): f32 accumulators that round once per 16 k here, 16 times a super-block in
place of 8, and one f32 rounding per share."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu

WHOLE = [((), 8192, 3072, 1000), ((), 7944, 768, 897), ((), 7937, 1280, 1001), ((), 8130, 512, 1024), ((), 6400, 1024, 1025), ((2,), 3840, 1536, 1000),
         ((), 16616, 512, 200), ((), 8184, 256, 2047)]
SHARED = [((), 2568, 10240, 513), ((), 3000, 8192, 1000), ((), 10984, 3072, 130)]


def operands(oracle, device, stack, m, k, n):
    rng = np.random.default_rng(m + k + n)
    s = stack[0] if stack else 1
    blocks = rng.integers(0, 256, (s * m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(s, m, k)).to("cuda:0")
    x = torch.from_numpy(rng.standard_normal((*stack, n, k)).astype(np.float16)).to("cuda:0")
    weight = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (*stack, m, k), device)
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(s, m, k // 256, 2)).to("cuda:0")
    bias = [torch.from_numpy(rng.standard_normal(l).astype(np.float16)).to("cuda:0") for l in (m, n)]
    xd = x.view(s, n, k).double()
    # the exact product, and what the two terms of a weight may reach before they cancel: 63 * 15 * d and 63 * dmin
    want = torch.stack([xd[i] @ w[i].T for i in range(s)])
    mag = torch.stack([xd[i].abs().view(n, -1, 256).sum(-1) @ (945 * sb[i, ..., 0] + 63 * sb[i, ..., 1]).T for i in range(s)]) + 2
    return weight, x, bias, want, mag


def tensor(v, device):
    return Tensor(tuple(v.shape), DType.F16, device, v.contiguous().view(torch.uint8).reshape(-1))


def bound(k):
    return 2.0**-24 * (k / 256 * 2 + 22 + 16)


@pytest.mark.parametrize("split,stack,m,k,n", [(split, *c) for c in WHOLE for split in (True, False)] + [(True, *c) for c in SHARED])
def test_edges(device, oracle, monkeypatch, split, stack, m, k, n):
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", split)
    s = stack[0] if stack else 1
    weight, x, bias, exact, mag = operands(oracle, device, stack, m, k, n)
    for to in (True, False):  # contiguous along the weight rows, and along the activations; the bias lies along the output's last axis
        for b in (bias[0 if to else 1], None):
            got = weight.gemm(tensor(x, device), None if b is None else tensor(b, device), False, True, to).resolve().storage.view(torch.float16)[: s * m * n]
            got = (got.view(s, n, m) if to else got.view(s, m, n).transpose(1, 2)).double()
            want = exact if b is None else exact + (b.double() if to else b.double()[:, None])
            err = (got - want).abs()
            assert (err <= 2.0**-11 * want.abs() + bound(k) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("act", ["gelu", "silu"])
@pytest.mark.parametrize("to", [True, False])
@pytest.mark.parametrize("m,k,n", [(7944, 768, 897), (7937, 1280, 1001)])  # rows of outputs that begin on 16 bytes (to), and that do not
def test_activation(device, oracle, m, k, n, to, act):
    weight, x, bias, exact, mag = operands(oracle, device, (), m, k, n)
    b = bias[0 if to else 1]
    got = getattr(weight.gemm(tensor(x, device), tensor(b, device), False, True, to), act)().resolve().storage.view(torch.float16)[: m * n]
    got = (got.view(n, m) if to else got.view(m, n).T).double()
    v = exact[0] + (b.double() if to else b.double()[:, None])
    want = v * torch.sigmoid(v if act == "silu" else 2 * v * (0.035677407 * v * v + 0.7978846))
    err = (got - want).abs()
    # 1.13: the largest slope of either; 2^-20: the exponential and the reciprocal
    assert (err <= (2.0**-11 + 2.0**-20) * want.abs() + 1.13 * bound(k) * mag[0] + 2.0**-25).all(), float((err / mag[0]).max())
