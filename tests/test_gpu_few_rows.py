"""3 to 16 activation rows against weights whose K is too long for the streaming matrix-core kernels (Q4_K and Q8_0H: the tiled kernels, K shared with a
workspace and whole without), and 5 to 8 rows against f16 weights of fewer than 128 tiles of 64 rows (launch_gemm_stream), against float64; and
plans that are given a workspace and none in turn.

The tolerance is that of the tiled kernels: products exact in f32, sums that round once per 16 or 32 k and share, the result rounded to f16."""
import ctypes

import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor, _ffi

pytestmark = pytest.mark.gpu


def weight(oracle, wt, m, k, rng):
    if wt == DType.Q4_K:
        blocks = rng.integers(0, 256, (m * k // 256, 144), dtype=np.uint8)
        blocks[:, :4] = (rng.uniform(0.5, 2, (len(blocks), 2)) / 1024).astype(np.float16).view(np.uint8)
        sb = blocks[:, :4].copy().view(np.float16).astype(np.float64).reshape(m, k // 256, 2)
        bound = np.repeat(945 * sb[..., 0] + 63 * sb[..., 1], 256, axis=1)  # what the two terms of a weight may reach before they cancel
        return blocks.reshape(-1), np.asarray(oracle.q4k_dequantize(blocks.reshape(-1)), dtype=np.float64).reshape(m, k), bound
    w = (rng.standard_normal((m, k)) / np.sqrt(k)).astype(np.float32)
    if wt == DType.F16:
        w = w.astype(np.float16)
        return w, w.astype(np.float64), np.abs(w.astype(np.float64))
    raw = oracle.make_q8_0h(w)
    codes = raw[: m * k].view(np.int8).reshape(m, k).astype(np.float64)
    off = (m * k + 255) // 256 * 256
    d = raw[off : off + m * k // 16].view(np.float16).astype(np.float64).reshape(m, k // 32)
    full = codes * np.repeat(d, 32, axis=1)
    return raw, full, np.abs(full)


CASES = [(DType.Q4_K, m, k, n) for m, k, n in [(1000, 4352, 9), (1280, 4352, 16), (70, 8448, 3), (1030, 8448, 8), (2560, 10240, 5), (640, 10240, 13), (64, 14336, 4)]] + [
    (DType.Q8_0H, m, k, n) for m, k, n in [(1280, 5120, 16), (1000, 8192, 9), (200, 10240, 5), (2560, 10240, 8), (1028, 10240, 16), (5120, 10240, 6), (640, 14336, 7)]] + [
    (DType.F16, m, k, n) for m, k, n in [(3072, 512, 5), (3200, 2560, 6), (4100, 1024, 8), (5536, 768, 7)]]


@pytest.mark.parametrize("split", [True, False])
@pytest.mark.parametrize("wt,m,k,n", CASES)
def test_against_float64(device, oracle, monkeypatch, wt, m, k, n, split):
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", split)
    rng = np.random.default_rng(m + k + n)
    raw, w, bound = weight(oracle, wt, m, k, rng)
    x, bias = rng.standard_normal((n, k)).astype(np.float16), rng.standard_normal(m).astype(np.float16)
    W = Tensor.from_data(raw, None, device) if wt == DType.F16 else Tensor.from_quantized(raw, wt, (m, k), device)
    got = W.gemm(Tensor.from_data(x, None, device), Tensor.from_data(bias, None, device), False, True, True).gelu().resolve().storage
    got = got.view(torch.float16)[: m * n].view(n, m).double()
    X = torch.from_numpy(x).to("cuda:0").double()
    want = X @ torch.from_numpy(w).to("cuda:0").T + torch.from_numpy(bias).to("cuda:0").double()
    mag = X.abs() @ torch.from_numpy(bound).to("cuda:0").T + 2
    z = want * (0.5 + 0.5 * torch.tanh(want * (0.035677407 * want * want + 0.7978846)))
    err = (got - z).abs()
    # 1.13: the largest slope of gelu; 2^-20: its exponential and reciprocal
    assert (err <= (2.0**-11 + 2.0**-20) * z.abs() + 1.13 * 2.0**-24 * (k / 16 / 8 + 40) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("wt,m,k,n", [(DType.Q4_K, 1000, 8448, 5), (DType.Q4_K, 1000, 4352, 12), (DType.Q8_0H, 1000, 10240, 6), (DType.Q8_0H, 1000, 8192, 12)])
def test_plan_with_and_without_workspace(device, oracle, wt, m, k, n):
    rng = np.random.default_rng(k + n)
    raw, _, _ = weight(oracle, wt, m, k, rng)
    L, W = _ffi.lib(), Tensor.from_quantized(raw, wt, (m, k), device)
    x = torch.randn((n, k), device="cuda:0").half()
    d, need, plan = _ffi.make_desc(wt, (m, k), DType.F16, (n, k), False, True, True), ctypes.c_uint64(), ctypes.c_void_p()
    assert L.rt_matmul_workspace_bytes(device.ctx, ctypes.byref(d), ctypes.byref(need)) == _ffi.RT_OK and need.value > 0
    ws = torch.empty(need.value, dtype=torch.uint8, device="cuda:0")
    assert L.rt_matmul_plan_create(device.ctx, ctypes.byref(d), 0, ctypes.byref(plan)) == _ffi.RT_OK
    stream = torch.cuda.current_stream().cuda_stream
    outs = []
    for use in (False, True, True, False, True, False):
        a, b = (torch.full((n, m), float("nan"), dtype=torch.float16, device="cuda:0") for _ in range(2))
        w, size = (ws.data_ptr(), need.value) if use else (None, 0)
        assert L.rt_matmul_plan_enqueue(plan, W.data_ptr(), x.data_ptr(), None, a.data_ptr(), w, size, stream) == _ffi.RT_OK
        assert L.rt_matmul_enqueue_ws(device.ctx, ctypes.byref(d), W.data_ptr(), x.data_ptr(), None, b.data_ptr(), 0, w, size, stream) == _ffi.RT_OK
        torch.cuda.synchronize()
        assert torch.equal(a, b) and a.isfinite().all()
        outs.append(a)
    assert torch.equal(outs[0], outs[3]) and torch.equal(outs[1], outs[4])
    L.rt_matmul_plan_destroy(plan)
