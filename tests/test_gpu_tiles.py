"""The tiled f16 and Q8_0H products (launch_gemm_nt): every tile and split its estimate chooses, at the edges of the tiles and for a K that
ends inside a tile of 64 or is no multiple of 256, against float64.

The tolerance: products of f16 numbers (and of codes) are exact in the MFMA, whose f32 accumulator rounds at most twice per 32 k, and a
Q8_0H block's sum is scaled and added with one more rounding, each by at most 2^-24 of the magnitudes summed; a shared K adds
its shares in at most 16 more; then the bias and the result's rounding to f16 (2^-11)."""
import numpy as np
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


def weights(device, gen, dt, stack, m, k):
    if dt == DType.F16:
        w = torch.randn((*stack, m, k), generator=gen, device="cuda:0").half()
        return tensor(device, w), w.double()
    n = m * k * (stack[0] if stack else 1)
    codes = torch.randint(-127, 128, (n,), generator=gen, device="cuda:0", dtype=torch.int8)
    scales = (torch.rand((n // 32,), generator=gen, device="cuda:0") * 0.02 + 1e-3).half()
    pad = lambda t: torch.nn.functional.pad(t.view(torch.uint8), (0, -t.view(torch.uint8).numel() % 256))
    w = Tensor((*stack, m, k), dt, device, torch.cat([pad(codes), pad(scales)]))
    return w, (codes.view(-1, 32).double() * scales.double()[:, None]).view(*stack, m, k)


def check(device, dt, m, n, k, trans_out=True, stack=()):
    gen = torch.Generator("cuda:0").manual_seed(m + n + k)
    w, wd = weights(device, gen, dt, stack, m, k)
    x, bias = (torch.randn(s, generator=gen, device="cuda:0").half() for s in ((*stack, n, k), (m,)))
    out = w.gemm(tensor(device, x), tensor(device, bias) if trans_out else None, False, True, trans_out).resolve()
    got = out.storage.view(torch.float16)[: out.numel()].view(out.shape).double()
    if not trans_out:
        got = got.transpose(-1, -2)
    b = bias.double() if trans_out else 0.0
    for lo in range(0, n, 512):
        xs = x[..., lo : lo + 512, :].double()
        wt = wd.transpose(-1, -2).contiguous()
        want, mag = xs @ wt + b, xs.abs() @ wt.abs() + (b.abs() if trans_out else 0.0)
        err = (got[..., lo : lo + 512, :] - want).abs()
        assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (3 * k / 32 + 20) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("m,n,k", [
    (333, 64, 288), (161, 7, 32), (200, 5, 96), (300, 65, 64), (4100, 130, 1056),                     # 64 x 64 tiles; one, two and more tiles of K
    (2051, 64, 4000), (1024, 33, 4128), (700, 300, 4064), (200, 9, 2080), (1000, 64, 8224),           # ... K shared, the last share shorter
    (5000, 300, 544), (2592, 512, 2592),                                                              # 64 x 128
    (9000, 200, 416), (20000, 100, 352),                                                              # 96 x 128
    (4090, 1001, 1440), (12800, 256, 320), (10241, 500, 288), (2560, 520, 10272),                     # 128 x 128, more than one round, K shared
    (10240, 512, 352), (20479, 511, 416), (10240, 512, 2592),                                         # 160 x 128
])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_k_of_whole_blocks(device, dt, m, n, k):
    check(device, dt, m, n, k)


@pytest.mark.parametrize("m,n,k", [(4480, 32, 4352), (4400, 40, 11008), (161, 9, 2816), (1027, 65, 4352), (2051, 33, 5888)])  # whole 256s, the last share shorter
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_unequal_shares(device, dt, m, n, k):
    check(device, dt, m, n, k)


@pytest.mark.parametrize("m", [4096, 4097, 4584, 4600])  # weight rows that fill the streaming kernel's grid, and the ones between that do not
@pytest.mark.parametrize("n,k", [(17, 1024), (32, 4096), (24, 4352)])
def test_few_rows_between_the_kernels(device, m, n, k):
    check(device, DType.Q8_0H, m, n, k)


@pytest.mark.parametrize("m,n,k", [(4352, 17, 4096), (4352, 32, 1024), (4352, 24, 4352), (4096, 20, 4096)])
def test_a_plan_gives_the_same_bits_whatever_workspace_came_before(device, m, n, k):
    """A plan offers its product first to the family that took it last; with and without a workspace it runs what a call without a plan does."""
    import ctypes

    from ratchet_amd import _ffi
    L, gen = _ffi.lib(), torch.Generator("cuda:0").manual_seed(m + n)
    w, _ = weights(device, gen, DType.Q8_0H, (), m, k)
    x = torch.randn((n, k), generator=gen, device="cuda:0").half()
    desc = _ffi.make_desc(_ffi.RT_Q8_0H, (m, k), _ffi.RT_F16, (1, n, k), False, True, True)
    need, plan = ctypes.c_uint64(), ctypes.c_void_p()
    assert L.rt_matmul_workspace_bytes(device.ctx, ctypes.byref(desc), ctypes.byref(need)) == _ffi.RT_OK
    ws = torch.empty(max(need.value, 16), dtype=torch.uint8, device="cuda:0")
    assert L.rt_matmul_plan_create(device.ctx, ctypes.byref(desc), _ffi.RT_ACT_NONE, ctypes.byref(plan)) == _ffi.RT_OK
    stream, ptrs = torch.cuda.current_stream().cuda_stream, (w.storage.data_ptr(), x.data_ptr(), None)
    try:
        for size in (need.value, 0, 0, need.value, need.value, 0):
            a, b = (torch.full((n, m), float("nan"), dtype=torch.float16, device="cuda:0") for _ in range(2))
            args = (ws.data_ptr() if size else None, size, stream)
            assert L.rt_matmul_plan_enqueue(plan, *ptrs, a.data_ptr(), *args) == _ffi.RT_OK
            assert L.rt_matmul_enqueue_ws(device.ctx, ctypes.byref(desc), *ptrs, b.data_ptr(), _ffi.RT_ACT_NONE, *args) == _ffi.RT_OK
            assert torch.equal(a, b), size
    finally:
        L.rt_matmul_plan_destroy(plan)


@pytest.mark.parametrize("m", [161, 162, 163, 164])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_sums_of_shares_of_any_row_length(device, dt, m):
    check(device, dt, m, 9, 4128)


@pytest.mark.parametrize("m,n,k", [
    (300, 300, 1024), (1024, 64, 4096), (200, 9, 8192), (2560, 512, 2304), (9000, 200, 512), (7681, 511, 512), (2560, 520, 10240), (10240, 512, 768),
])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_k_of_whole_units(device, dt, m, n, k):
    check(device, dt, m, n, k)


@pytest.mark.parametrize("m,n,k", [  # the smallest numbers of activation rows that leave the streaming kernels, on both sides of the line
    (8192, 5, 288), (8100, 5, 288), (8129, 8, 544), (8128, 8, 544), (9000, 4, 288), (16400, 7, 352), (4097, 17, 512), (4032, 17, 512), (5120, 32, 1024)])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_few_activation_rows(device, dt, m, n, k):
    check(device, dt, m, n, k)


@pytest.mark.parametrize("m,n,k", [(333, 70, 288), (1001, 300, 800), (2600, 130, 4000)])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_other_axis_contiguous(device, dt, m, n, k):
    check(device, dt, m, n, k, trans_out=False)


@pytest.mark.parametrize("stacks,m,n,k", [(3, 200, 33, 288), (2, 700, 130, 2080), (5, 161, 9, 1056), (2, 300, 70, 512)])
@pytest.mark.parametrize("dt", [DType.Q8_0H, DType.F16])
def test_stacks(device, dt, stacks, m, n, k):
    check(device, dt, m, n, k, trans_out=False, stack=(stacks,))


def test_scales_at_the_end_of_the_stream(device):
    """Rows whose last scales are the stream's last bytes: 8 blocks too many are asked for at every offset from its end."""
    for m in range(160, 168):
        for k in (32, 64, 96, 288, 352):
            check(device, DType.Q8_0H, m, 9, k)


@pytest.mark.parametrize("dt,m,n,k", [(DType.Q8_0H, 700, 300, 4064), (DType.F16, 2051, 64, 4000), (DType.Q8_0H, 2560, 520, 10240)])
def test_without_a_workspace(device, monkeypatch, dt, m, n, k):
    import ratchet_amd.tensor as mirror
    monkeypatch.setattr(mirror, "SPLIT_K", False)
    check(device, dt, m, n, k)
