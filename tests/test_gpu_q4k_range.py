"""Q4_K products over the range of f16 activations: 32 of one sign sum to up to 32 x 65504, which the kernels hold as f16 parts, and small ones to f16
subnormals.  Against float64, at the sizes of each kernel that does so, with a workspace and without.

The tolerance is that of the other Q4_K tests: f32 accumulators that round once per 16 or 32 k and share, sums of x that round once per addition and to
23 bits as parts, all relative to what the two terms of a weight may reach before they cancel, and the f16 rounding of the output."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu

FEW = [(70, 8448, 3), (1030, 8448, 8), (1000, 4352, 9), (640, 10240, 16)]  # K shared, and whole without a workspace
PREFILL = [(3072, 512, 64), (8192, 512, 200), (8192, 768, 300)]  # one and two weight tiles per wavefront, with and without loading wavefronts
STREAM = [(520, 1024, 1), (520, 4096, 2), (512, 8192, 4), (1030, 5120, 8), (512, 4096, 16), (8192, 512, 16), (1030, 768, 29)]  # gemv_q4k_mfma_kernel
WIDE = [(8192, 768, 1000), (7937, 1280, 1001)]  # gemm_q4k_wide_kernel


def product(oracle, device, m, k, n, x, d_exp, seed):
    """got, want and the magnitudes of the terms, for weights d * sc * q - dmin * mn of d about 2^d_exp and terms of one size."""
    rng = np.random.default_rng(seed)
    blocks = rng.integers(0, 256, (m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) * np.array([2.0**d_exp, 2.0 ** (d_exp + 3)])).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(m, k)).to("cuda:0")
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(m, k // 256, 2)).to("cuda:0")
    X = torch.from_numpy(x).to("cuda:0")
    t = Tensor((n, k), DType.F16, device, X.view(torch.uint8).reshape(-1))
    got = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (m, k), device).gemm(t, None, False, True, True).resolve()
    got = got.storage.view(torch.float16)[: m * n].view(n, m).double()
    mag = X.double().abs().view(n, -1, 256).sum(-1) @ (945 * sb[..., 0] + 63 * sb[..., 1]).T
    return got, X.double() @ w.T, mag


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("size,d_exp", [(5000.0, -18), (65504.0, -22), (2.0**-14, -2)])
@pytest.mark.parametrize("m,k,n", FEW + PREFILL + WIDE + STREAM)
def test_one_sign_per_block(device, oracle, monkeypatch, m, k, n, size, d_exp, split):
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", split)
    rng = np.random.default_rng(m + k + n)
    sign = np.repeat(rng.choice([-1.0, 1.0], (n, k // 32)), 32, axis=1)
    x = (sign * rng.uniform(0.9, 1.0, (n, k)) * size).astype(np.float16)
    got, want, mag = product(oracle, device, m, k, n, x, d_exp, m + k)
    assert want.abs().max() < 60000  # (in f16)
    err = (got - want).abs()
    assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 256 * 2 + 54) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("stack,m,k,n", [((), 70, 8448, 3), ((), 2560, 10240, 5), ((), 1030, 8448, 8), ((2,), 130, 14336, 4)])
def test_infinite_activation(device, oracle, monkeypatch, stack, m, k, n, bias, split):
    """3 to 8 rows: a weight times an infinity is one, of its sign, with a workspace and without; the other rows' outputs are what they would be."""
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", split)
    rng = np.random.default_rng(m + k + n)
    s = stack[0] if stack else 1
    blocks = rng.integers(0, 256, (s * m * k // 256, 144), dtype=np.uint8)
    blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
    w = torch.from_numpy(np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(s, m, k)).to("cuda:0")
    sb = torch.from_numpy(blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(s, m, k // 256, 2)).to("cuda:0")
    x = rng.standard_normal((*stack, n, k)).astype(np.float16)
    x.reshape(s, n, k)[0, 1, 777] = np.inf
    x.reshape(s, n, k)[s - 1, n - 1, [0, k - 1]] = -np.inf, np.inf
    X, b = torch.from_numpy(x).to("cuda:0"), torch.from_numpy(rng.standard_normal(m).astype(np.float16)).to("cuda:0")
    t = lambda v: Tensor(tuple(v.shape), DType.F16, device, v.contiguous().view(torch.uint8).reshape(-1))
    W = Tensor.from_quantized(blocks.reshape(-1), DType.Q4_K, (*stack, m, k), device)
    for to in (True, False):
        got = W.gemm(t(X), t(b) if bias and to else None, False, True, to).resolve().storage.view(torch.float16)[: s * m * n]
        got = (got.view(s, n, m) if to else got.view(s, m, n).transpose(1, 2)).double()
        for i in range(s):
            xd = X.view(s, n, k)[i].double()
            want = (xd[:, None, :] * w[i][None]).sum(-1) + (b.double() if bias and to else 0)
            finite = xd.isfinite().all(1)
            mag = xd.abs().view(n, -1, 256).sum(-1) @ (945 * sb[i, ..., 0] + 63 * sb[i, ..., 1]).T + 2
            err = (got[i] - want).abs()
            assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 256 * 2 + 54) * mag + 2.0**-25)[finite].all()
            special = ~finite
            assert int(special.sum()) == len({(0, 1), (s - 1, n - 1)} & {(i, j) for j in range(n)})
            assert torch.equal(got[i][special].isnan(), want[special].isnan())
            assert torch.equal(got[i][special].nan_to_num(0.0), want[special].nan_to_num(0.0)) and not got[i][special].isfinite().any()
