"""Q4_K weights against many activation rows with K shared among workgroups (launch_gemm_q4k with a workspace): shares of one and more
super-blocks, the last one shorter, tiles that end inside the weight and the activations, stacks, and the same products with K whole,
against float64.

The tolerance: that of the unshared kernel (f32 accumulators that round once per 32 k, d and dmin applied in f32 per super-block, sums of x
held to 2^-22, the result rounded to f16 once) and one f32 rounding per share."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("stack,m,k,n", [
    ((), 2560, 10240, 64), ((), 3072, 8192, 33), ((), 1000, 4096, 129), ((), 828, 1280, 70), ((), 100, 3328, 19), ((), 3584, 9472, 148),
    ((), 64, 2560, 1000), ((3,), 320, 2816, 65), ((2,), 1090, 5120, 40)])
def test_shares(device, oracle, monkeypatch, stack, m, k, n, split):
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
            assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 256 * 2 + 14 + 16) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("m,n,k,shared", [(2560, 32, 4096, False), (2560, 17, 2560, False), (2560, 33, 4096, True), (2560, 32, 4352, True),
                                          (5000, 32, 2560, False), (5000, 17, 4096, True)])
def test_workspace_only_where_the_shares_run(device, m, n, k, shared):
    """Up to 32 activation rows run on the streaming kernel, which shares nothing, as far as its LDS goes."""
    import ctypes

    from ratchet_amd import _ffi
    need = ctypes.c_uint64()
    d = _ffi.make_desc(_ffi.RT_Q4_K, (m, k), _ffi.RT_F16, (1, n, k), False, True, True)
    assert _ffi.lib().rt_matmul_workspace_bytes(device.ctx, ctypes.byref(d), ctypes.byref(need)) == _ffi.RT_OK
    assert (need.value > 0) == shared
