"""Q8_0F weights against 1 to 8 f32 vectors (gemv_q8f_kernel): weight rows that end inside a workgroup's four, K that ends inside a step of 256 and inside
the four wavefronts' steps, stacks, both orders of the output, bias along either axis, infinities, against float64.

The tolerance: a product is rounded once, four of them and their scale's make five roundings, a lane adds one sum per 1024 k, and ten additions
join the lanes and wavefronts: 2^-24 of the magnitudes for each, and one for the bias.  The limb kernel adds a sum per MFMA of 32 k."""
import ctypes

import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor, _ffi

pytestmark = pytest.mark.gpu


def make(m, k, rng, s=1):
    codes = rng.integers(-128, 128, (s * m, k), dtype=np.int8)
    d = rng.uniform(0.5, 2, (s * m, k // 32)).astype(np.float32) / 128
    pad = lambda b: np.concatenate([b, np.zeros(-len(b) % 256, np.uint8)])
    raw = np.concatenate([pad(codes.reshape(-1).view(np.uint8)), pad(d.reshape(-1).view(np.uint8))])
    return raw, codes.astype(np.float64) * np.repeat(d.astype(np.float64), 32, axis=1)


@pytest.mark.parametrize("n", range(1, 9))
@pytest.mark.parametrize("stack,m,k", [((), 1, 32), ((), 3, 96), ((), 5, 256), ((), 1001, 288), ((), 66, 1024), ((), 7, 1056), ((), 130, 4128), ((3,), 9, 640)])
def test_against_float64(device, stack, m, k, n):
    rng = np.random.default_rng(m + k + n)
    s = stack[0] if stack else 1
    raw, w = make(m, k, rng, s)
    w = w.reshape(s, m, k)
    x, bias = rng.standard_normal((*stack, n, k)).astype(np.float32), rng.standard_normal(m).astype(np.float32)
    W, X = Tensor.from_quantized(raw, DType.Q8_0F, (*stack, m, k), device), Tensor.from_data(x, None, device)
    for to in (True, False):
        b = bias if to else rng.standard_normal(n).astype(np.float32)
        got = W.gemm(X, Tensor.from_data(b, None, device), False, True, to).resolve().storage.view(torch.float32)[: s * m * n].cpu().numpy().astype(np.float64)
        got = got.reshape(s, n, m) if to else got.reshape(s, m, n).transpose(0, 2, 1)
        for i in range(s):
            xd = x.reshape(s, n, k)[i].astype(np.float64)
            want = xd @ w[i].T + (b[None, :] if to else b[:, None])
            mag = np.abs(xd) @ np.abs(w[i]).T
            assert (np.abs(got[i] - want) <= 2.0**-24 * ((k / 1024 + 16) * mag + np.abs(want))).all(), (np.abs(got[i] - want) / mag).max() * 2**24


@pytest.mark.parametrize("n", (9, 15, 16, 17))
@pytest.mark.parametrize("m,k", [(1, 1024), (4096, 1024), (4097, 1024), (33, 992), (1279, 4096), (1281, 4096), (130, 4128)])
def test_two_launches(device, m, k, n):
    """9 to 16 vectors go in two launches at K >= 1024, up to 4096 rows and 5 x 2^20 codes: on both sides of each of these, the vectors also 4 bytes past an
    aligned address."""
    rng = np.random.default_rng(m + k + n)
    raw, w = make(m, k, rng)
    x, bm, bn = (rng.standard_normal(s).astype(np.float32) for s in ((n, k), m, n))
    W = Tensor.from_quantized(raw, DType.Q8_0F, (m, k), device)
    room = torch.zeros(4 * n * k + 16, dtype=torch.uint8, device="cuda:0")
    room[4 : 4 + 4 * n * k] = torch.from_numpy(x.view(np.uint8).reshape(-1)).to("cuda:0")
    xd = x.astype(np.float64)
    mag = np.abs(xd) @ np.abs(w).T
    for X in (Tensor.from_data(x, None, device), Tensor((n, k), DType.F32, device, room[4 : 4 + 4 * n * k])):
        for to in (True, False):
            got = W.gemm(X, Tensor.from_data(bm if to else bn, None, device), False, True, to).resolve().storage.view(torch.float32)[: m * n].cpu().numpy().astype(np.float64)
            got, want = (got.reshape(n, m), xd @ w.T + bm[None, :]) if to else (got.reshape(m, n).T, xd @ w.T + bn[:, None])
            assert (np.abs(got - want) <= 2.0**-24 * ((k / 32 + 16) * mag + np.abs(want))).all(), (np.abs(got - want) / mag).max() * 2**24


def test_infinite_activation(device):
    """Only the outputs of its vector are touched, also where it stands past another lane's end of the row."""
    raw, w = make(10, 288, np.random.default_rng(1))
    x = np.ones((3, 288), np.float32)
    x[1, 287] = np.inf
    out = Tensor.from_quantized(raw, DType.Q8_0F, (10, 288), device).gemm(Tensor.from_data(x, None, device), None, False, True, True).resolve()
    out = out.storage.view(torch.float32)[:30].view(3, 10).cpu().numpy()
    assert np.isfinite(out[[0, 2]]).all() and (out[1] == np.where(w[:, 287] == 0, np.nan, np.sign(w[:, 287]) * np.inf))[w[:, 287] != 0].all()


@pytest.mark.parametrize("n", (1, 2))
def test_more_rows_than_one_launch(device, n):
    """A launch's threads number less than 2^32, 2^24 - 1 workgroups of four rows: the rows beyond go in a second one.  On both sides of that, and at either end."""
    m, k = 2**26 + 5, 32
    gen = torch.Generator("cuda:0").manual_seed(n)
    codes = torch.empty((m, k), dtype=torch.int8, device="cuda:0").random_(-127, 128, generator=gen)
    d = torch.rand(m, generator=gen, device="cuda:0") / 64 + 2.0**-8
    pad = lambda b: torch.nn.functional.pad(b.view(torch.uint8).reshape(-1), (0, -b.numel() * b.element_size() % 256))
    x, bias = torch.randn((n, k), generator=gen, device="cuda:0"), torch.randn(m, generator=gen, device="cuda:0")
    t = lambda v, shape, dt=DType.F32: Tensor(shape, dt, device, v.contiguous().view(torch.uint8).reshape(-1))
    got = t(torch.cat([pad(codes), pad(d)]), (m, k), DType.Q8_0F).gemm(t(x, (n, k)), t(bias, (m,)), False, True, True).resolve().storage.view(torch.float32)[: m * n].view(n, m)
    assert got.isfinite().all()
    edge = 4 * (2**24 - 1)
    for rows in (slice(0, 64), slice(edge - 64, edge + 64), slice(m - 64, m)):
        w = codes[rows].double() * d[rows].double()[:, None]
        want, mag = x.double() @ w.T + bias[rows].double(), x.double().abs() @ w.abs().T
        assert ((got[:, rows] - want).abs() <= 2.0**-24 * (16 * mag + want.abs())).all()


@pytest.mark.parametrize("n", (1, 2, 5, 8, 9, 16))
def test_vectors_at_any_address(device, n):
    """One kernel whatever 4-byte address the vectors start at, for which no workspace is asked: the same bits as on an aligned one."""
    m, k = 1003, 1056
    rng = np.random.default_rng(n)
    raw, _ = make(m, k, rng)
    x = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to("cuda:0")
    W = Tensor.from_quantized(raw, DType.Q8_0F, (m, k), device)
    outs = []
    for at in (0, 4, 8, 12, 20):
        room = torch.zeros(4 * n * k + 32, dtype=torch.uint8, device="cuda:0")
        room[at : at + 4 * n * k] = x.view(torch.uint8).reshape(-1)
        out = W.gemm(Tensor((n, k), DType.F32, device, room[at : at + 4 * n * k]), None, False, True, True).resolve()
        outs.append(out.storage.view(torch.float32)[: m * n].clone())
    assert outs[0].isfinite().all() and all(torch.equal(outs[0], o) for o in outs[1:])


@pytest.mark.parametrize("m,k,n,asks", [(1001, 4096, 8, False), (1001, 4096, 9, False), (1001, 4096, 16, False), (1001, 4096, 17, True), (1001, 992, 16, True), (4097, 1024, 16, True)])
def test_workspace_only_where_it_is_used(device, m, k, n, asks):
    d, need = _ffi.make_desc(DType.Q8_0F, (m, k), DType.F32, (n, k), False, True, True), ctypes.c_uint64()
    assert _ffi.lib().rt_matmul_workspace_bytes(device.ctx, ctypes.byref(d), ctypes.byref(need)) == _ffi.RT_OK
    assert (need.value > 0) == asks
