"""f32 products on the bf16 matrix cores (kernels_gemm_limb.hip) at the sizes and values where they can go wrong, against
float64.

The tolerance is the rounding of the accumulation: a sum of K products takes at most six MFMAs per 16 k, each of which rounds
the accumulator once, plus the fold of a block, the sum over the shares of K and the bias, every rounding at most 2^-24 of
the magnitudes summed."""
import math

import numpy as np
import pytest
import torch

from ratchet_amd import DType, Device, Tensor, Quantization, Quantizer, dequantize

pytestmark = pytest.mark.gpu


def bound(x, y, bias):
    k = x.shape[-1]
    mag = np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64)
    return 2.0**-24 * (6 * (k / 16 + 1) + 4) * (mag + (0 if bias is None else np.abs(bias)))


def run(device, a, b, bias, tl, tr, to):
    t = lambda v: None if v is None else Tensor.from_data(v).to(device)
    return t(a).gemm(t(b), t(bias), tl, tr, to).resolve().to(Device.CPU).storage


@pytest.mark.parametrize("tl,tr,to", [(False, False, False), (True, False, False), (False, True, False), (True, False, True), (False, True, True)])
@pytest.mark.parametrize("stacks,m,k,n", [
    (1, 65, 65, 129), (1, 97, 1500, 64), (3, 130, 99, 70), (1, 1500, 68, 33), (1, 16, 2049, 300), (1, 40, 3001, 40), (7, 300, 65, 301),
    (1, 9, 66, 20001), (40, 129, 64, 130), (1, 2000, 96, 1999)])
def test_layouts_and_edges(device, stacks, m, k, n, tl, tr, to):
    rng = np.random.default_rng(m * 7 + k)
    x, y = rng.standard_normal((stacks, m, k)).astype(np.float32), rng.standard_normal((stacks, k, n)).astype(np.float32)
    bias = rng.standard_normal(m if to else n).astype(np.float32) if stacks == 1 else None
    got = run(device, np.swapaxes(x, 1, 2) if tl else x, np.swapaxes(y, 1, 2) if tr else y, bias, tl, tr, to)
    b = 0 if bias is None else bias[:, None] if to else bias
    want = x.astype(np.float64) @ y.astype(np.float64) + b
    err = np.abs((np.swapaxes(got, 1, 2) if to else got) - want)
    assert (err <= bound(x, y, None if bias is None else b)).all(), (err / bound(x, y, None if bias is None else b)).max()


@pytest.mark.parametrize("rows,n,k", [(9, 33, 64), (17, 127, 96), (65, 129, 32), (129, 257, 320), (200, 2560, 10240), (300, 100, 4096), (13, 20000, 288)])
@pytest.mark.parametrize("swap", [False, True])
def test_codes_with_f32_scales(device, rows, n, k, swap):
    rng = np.random.default_rng(rows + k)
    w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data(rng.standard_normal((n, k)).astype(np.float32)).to(device))
    x = rng.standard_normal((rows, k)).astype(np.float32)
    wf = dequantize(w).to(Device.CPU).storage
    bias = rng.standard_normal(n if not swap else n).astype(np.float32)
    xt, bt = Tensor.from_data(x).to(device), Tensor.from_data(bias).to(device)
    if swap:  # out [n, rows], whose contiguous axis is the activations': no bias there
        got = w.gemm(xt, None, False, True, False).resolve().to(Device.CPU).storage.T
        bias = np.zeros_like(bias)
    else:
        got = w.gemm(xt, bt, False, True, True).resolve().to(Device.CPU).storage
    want = x.astype(np.float64) @ wf.astype(np.float64).T + bias
    assert (np.abs(got - want) <= bound(x, wf.T, bias)).all()


@pytest.mark.parametrize("scale_x,scale_y", [(1e-36, 1e3), (1e18, 1e18), (1e-20, 1e-15), (1e30, 1e-30)])
def test_magnitudes(device, scale_x, scale_y):
    """Limbs of small numbers reach into bf16's subnormals; results leave the range of f32 at either end."""
    rng = np.random.default_rng(3)
    x, y = (rng.standard_normal((70, 200)) * scale_x).astype(np.float32), (rng.standard_normal((200, 90)) * scale_y).astype(np.float32)
    got = run(device, x, y, None, False, False, False)
    want = x.astype(np.float64) @ y.astype(np.float64)
    with np.errstate(over="ignore"):
        inside = np.abs(want) < 3e38
    # the last limb is a multiple of bf16's smallest subnormal number, 2^-133: half of that of the other operand per product;
    # and the results' own subnormals
    tiny = 2.0**-134 * (np.abs(y).sum(0)[None, :] + np.abs(x).sum(1)[:, None]) + 200 * 2.0**-149
    assert (np.abs(got - want) <= bound(x, y, None) + tiny)[inside].all()
    assert np.isinf(got[np.abs(want) > 4e38]).all()


def test_values_that_are_not_finite(device):
    """What the f32 arithmetic gives: infinities of either sign, NaN from inf - inf, inf * 0 and NaN operands, numbers that
    round past the largest bf16."""
    rng = np.random.default_rng(4)
    x, y = rng.standard_normal((130, 160)).astype(np.float32), rng.standard_normal((160, 140)).astype(np.float32)
    x[3, 5], x[7, 0], x[9, 9], x[9, 10] = np.inf, -np.inf, np.inf, -np.inf
    x[20, 159], x[64, 31], y[8, 60], y[5, 100] = np.nan, 3.4e38, np.inf, 0.0
    y[31, 2] = 0.25
    for trans in (False, True):
        got = run(device, x, y.T.copy() if trans else y, None, False, trans, False)
        with np.errstate(invalid="ignore", over="ignore"):
            want = (x.astype(np.float64) @ y.astype(np.float64)).astype(np.float32)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
        fine = np.isfinite(want)
        assert np.isfinite(got[fine]).all() and np.allclose(got[fine], want[fine], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("m", [65535 * 64, 65535 * 64 + 1, 65536 * 64 + 65])
def test_rows_beyond_one_grid(device, m):
    """Strides of millions of values are the generic kernel's, whose 65535 tiles along a grid's second axis hold 4.2 million rows."""
    gen = torch.Generator("cuda:0").manual_seed(m)
    x, y = torch.randn((3, m), generator=gen, device="cuda:0"), torch.randn((3, 20), generator=gen, device="cuda:0")
    t = lambda v: Tensor(tuple(v.shape), DType.F32, device, v.view(torch.uint8).reshape(-1))
    got = t(x).gemm(t(y), None, True, False, False).resolve().storage.view(torch.float32)[: 20 * m].view(m, 20)
    for lo in range(0, m, 1 << 20):  # three products, at most three roundings
        xd = x[:, lo : lo + (1 << 20)].double().T.contiguous()
        err = (got[lo : lo + (1 << 20)].double() - xd @ y.double()).abs()
        assert (err <= 2.0**-24 * 4 * (xd.abs() @ y.double().abs()) + 2.0**-149).all()


@pytest.mark.parametrize("tl", [False, True])
@pytest.mark.parametrize("k,n", [(65, 9), (96, 63), (96, 64), (200, 65), (300, 127), (511, 128), (65, 129), (600, 300), (3001, 131), (70, 20001)])
def test_one_row_written_as_a_column(device, monkeypatch, k, n, tl):
    """[1, K] . [K, N] with the output transposed: both strides of the output are 1, and rows past the only one must not be
    stored.  With and without K shared."""
    rng = np.random.default_rng(k + n)
    x, y = rng.standard_normal((1, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    want, b = x.astype(np.float64) @ y.astype(np.float64), bound(x, y, None)
    for share in (True, False):
        monkeypatch.setattr("ratchet_amd.tensor.SPLIT_K", share)
        got = run(device, x.T.copy() if tl else x, y, None, tl, False, True)
        assert got.shape == (n, 1) and (np.abs(got.T - want) <= b).all(), (share, (np.abs(got.T - want) / b).max())


@pytest.mark.parametrize("n,k", [(33, 64), (300, 96), (1000, 4096)])
def test_codes_against_one_misaligned_row(device, n, k):
    """One activation row that the streaming kernels do not take (4 bytes past a 16-byte boundary), the output [N, 1]."""
    rng = np.random.default_rng(n + k)
    w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data(rng.standard_normal((n, k)).astype(np.float32)).to(device))
    x = rng.standard_normal((k, 1)).astype(np.float32)
    room = torch.zeros(4 * k + 16, dtype=torch.uint8, device="cuda:0")
    room[4 : 4 + 4 * k] = torch.from_numpy(x.view(np.uint8).reshape(-1)).to("cuda:0")
    xt = Tensor((k, 1), DType.F32, device, room[4 : 4 + 4 * k])
    wf = dequantize(w).to(Device.CPU).storage
    got = w.gemm(xt, None, False, False, False).resolve().to(Device.CPU).storage
    assert got.shape == (n, 1) and (np.abs(got - wf.astype(np.float64) @ x.astype(np.float64)) <= bound(x.T, wf.T, None).T).all()


@pytest.mark.parametrize("tr", [False, True])
@pytest.mark.parametrize("stacks,m,k,n", [
    (32, 512, 4, 512), (3, 2041, 32, 2044), (20, 300, 28, 300),  # one K tile: 128 x 128 tiles, ragged ones, the small tiles
    (1, 520, 32, 48), (8, 128, 128, 128), (1, 96, 132, 96),      # few tiles: up to K = 128 and past it
    (16, 100, 100, 64), (1, 1536, 508, 52), (1, 1536, 512, 52), (1, 300, 384, 64)])
def test_small_products_on_either_side_of_the_rules(device, stacks, m, k, n, tr):
    """Products that stay on the f32 matrix cores (launch_gemm_f32_small) and the first ones past them."""
    rng = np.random.default_rng(m + k + n)
    x, y = rng.standard_normal((stacks, m, k)).astype(np.float32), rng.standard_normal((stacks, k, n)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    got = run(device, x, np.swapaxes(y, 1, 2) if tr else y, bias, False, tr, False)
    want = x.astype(np.float64) @ y.astype(np.float64) + bias
    # the f32 matrix cores round after each product
    assert (np.abs(got - want) <= 2.0**-24 * (k + 2) * (np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64) + np.abs(bias))).all()


@pytest.mark.parametrize("tl,tr", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("stacks,m,n", [(1, 1100, 1029), (32, 512, 512), (1, 70, 90)])
def test_outer_products_are_rounded_once(device, stacks, m, n, tl, tr):
    """K = 1: every output is the correctly rounded product.  K = 2: the sum of two products is rounded twice."""
    rng = np.random.default_rng(m + n)
    for k in (1, 2):
        x, y = rng.standard_normal((stacks, m, k)).astype(np.float32), rng.standard_normal((stacks, k, n)).astype(np.float32)
        got = run(device, np.swapaxes(x, 1, 2) if tl else x, np.swapaxes(y, 1, 2) if tr else y, None, tl, tr, False)
        want = x.astype(np.float64) @ y.astype(np.float64)
        if k == 1:
            assert np.array_equal(got, want.astype(np.float32))
        else:
            assert (np.abs(got - want) <= 2.0**-24 * (np.abs(x[..., :1].astype(np.float64) * y[:, :1]) + np.abs(got)) * (1 + 2.0**-20)).all()


def close_or_alike(got, want, b):
    """Within the bound where the result is finite; the same infinities and NaNs where it is not."""
    fine = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    assert (np.abs(got[fine].astype(np.float64) - want[fine]) <= b[fine] + 2.0**-24 * np.abs(want[fine])).all()


@pytest.mark.parametrize("tl,tr,to", [(False, False, False), (True, False, False), (False, True, False), (True, True, False), (False, True, True), (True, False, True)])
@pytest.mark.parametrize("m,k,n", [(130, 68, 70), (200, 99, 260), (64, 1055, 96), (70, 2049, 90), (1, 150, 90), (1500, 96, 1500)])
def test_products_computed_once_more(device, m, k, n, tl, tr, to):
    """Rows and columns that are not finite and numbers past the largest bf16, in every layout, K shared and not, with ragged K: a
    tile that holds one is computed again and its finite outputs stay what they are."""
    rng = np.random.default_rng(m + k + n)
    x, y = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    bias = rng.standard_normal(m if to else n).astype(np.float32)
    x[m // 2], x[m - 1, k - 1], y[k - 1, n // 3] = np.nan, np.inf, -np.inf
    x[0, 0], y[0] = 3.4e38, rng.choice([-0.25, 0.0, 0.5], n).astype(np.float32)  # the limbs of the first are not finite, the product is
    got = run(device, x.T.copy() if tl else x, y.T.copy() if tr else y, bias, tl, tr, to)
    with np.errstate(invalid="ignore", over="ignore"):
        b = bias[:, None] if to else bias
        want = (x.astype(np.float64) @ y.astype(np.float64) + b).astype(np.float32)
        # computed again: rounded after each product
        limit = 2.0**-24 * (k + 6) * (np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64) + np.abs(b))
    close_or_alike(got.T if to else got, want, limit)


@pytest.mark.parametrize("to", [True, False])
@pytest.mark.parametrize("rows,n,k", [(33, 100, 64), (200, 257, 96), (200, 2560, 2560), (20, 40, 4096)])
def test_codes_computed_once_more(device, rows, n, k, to):
    """The same against Q8_0F weights with a scale that is infinite, in both orders of the output, with a bias on either axis."""
    rng = np.random.default_rng(rows + k)
    w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data(rng.standard_normal((n, k)).astype(np.float32)).to(device))
    scales = w.storage[(n * k + 255) // 256 * 256 :].view(torch.float32)
    scales[(n // 2) * (k // 32) + k // 32 - 1] = math.inf
    codes = w.storage[: n * k].view(torch.int8).cpu().numpy().reshape(n, k)
    with np.errstate(invalid="ignore"):
        wf = codes * np.repeat(scales[: n * k // 32].cpu().numpy().reshape(n, -1), 32, axis=1)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x[rows // 2], x[rows - 1, 0] = np.nan, 3.4e38
    wf[:, 0] = np.where(codes[:, 0] == 0, 0.0, wf[:, 0])
    bias = rng.standard_normal(n if to else rows).astype(np.float32)
    t = lambda v: Tensor.from_data(v).to(device)
    got = w.gemm(t(x), t(bias), False, True, to).resolve().to(Device.CPU).storage
    with np.errstate(invalid="ignore", over="ignore"):
        b = bias if to else bias[:, None]
        want = (x.astype(np.float64) @ wf.astype(np.float64).T + b).astype(np.float32)
        limit = 2.0**-24 * (2 * k + 6) * (np.abs(x).astype(np.float64) @ np.abs(wf).astype(np.float64).T + np.abs(b))
    close_or_alike(got if to else got.T, want, limit)


@pytest.mark.parametrize("tr", [False, True])
@pytest.mark.parametrize("scale_x,scale_y", [(1e-34, 1e3), (1e-36, 1e3), (1e-38, 1e5), (1e-40, 1e10), (1e-43, 1e20), (1e-36, 1e36), (1e-20, 1e-15), (1e34, 1e-38)])
def test_small_numbers_keep_their_digits(device, scale_x, scale_y, tr):
    """Every f32 number is the exact sum of its limbs, down to f32's subnormal ones; what is left is the rounding of the sums and
    of results that are subnormal."""
    rng = np.random.default_rng(5)
    x, y = (rng.standard_normal((150, 200)) * scale_x).astype(np.float32), (rng.standard_normal((200, 290)) * scale_y).astype(np.float32)
    got = run(device, x, y.T.copy() if tr else y, None, False, tr, False)
    want = x.astype(np.float64) @ y.astype(np.float64)
    assert (np.abs(got - want) <= bound(x, y, None) + 2.0**-149).all()


def test_small_activations_against_codes_keep_their_digits(device):
    rng = np.random.default_rng(6)
    for scale_x, scale_w in ((1e-36, 1.0), (1e-41, 1e6), (1e-3, 1e-37), (1e20, 1e-37)):
        w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data((rng.standard_normal((140, 96)) * scale_w).astype(np.float32)).to(device))
        wf = w.storage[: 140 * 96].view(torch.int8).double().view(-1, 32) * w.storage[(140 * 96 + 255) // 256 * 256 :].view(torch.float32)[: 140 * 3].double()[:, None]
        wf = wf.view(140, 96).cpu().numpy()
        x = (rng.standard_normal((40, 96)) * scale_x).astype(np.float32)
        got = w.gemm(Tensor.from_data(x).to(device), None, False, True, True).resolve().to(Device.CPU).storage
        assert (np.abs(got - x.astype(np.float64) @ wf.T) <= bound(x, wf.T, None) + 4 * 2.0**-149).all()


@pytest.mark.parametrize("tl,tr", [(False, False), (False, True), (True, False)])
def test_every_limb_counts(device, tl, tr):
    """One product per output: six MFMAs make it, the last one's sum is cut at 2^-23 of it, and what the sums before it and the products
    left out (2^-26) miss is less than that.  Without any one limb product 2^-18 of it would be missing."""
    rng = np.random.default_rng(7)
    for m, k, n in ((300, 96, 300), (130, 2048, 70), (1500, 68, 1500)):
        x, y = np.zeros((m, k), np.float32), rng.standard_normal((k, n)).astype(np.float32)
        at = rng.integers(0, k, m)
        x[np.arange(m), at] = rng.standard_normal(m)
        got = run(device, x.T.copy() if tl else x, y.T.copy() if tr else y, None, tl, tr, False)
        want = x[np.arange(m), at].astype(np.float64)[:, None] * y[at]
        assert (np.abs(got - want) <= 4 * 2.0**-24 * np.abs(want)).all(), (np.abs(got - want) / np.abs(want)).max() * 2**24


def test_every_limb_counts_against_codes(device):
    """Three MFMAs make a product of an activation and a code, and the fold with the scale rounds once more."""
    rng = np.random.default_rng(8)
    n, k, rows = 300, 96, 200
    w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data(rng.standard_normal((n, k)).astype(np.float32)).to(device))
    wf = (w.storage[: n * k].view(torch.int8).double().view(-1, 32) * w.storage[(n * k + 255) // 256 * 256 :].view(torch.float32)[: n * k // 32].double()[:, None])
    wf = wf.view(n, k).cpu().numpy()
    x, at = np.zeros((rows, k), np.float32), rng.integers(0, k, rows)
    x[np.arange(rows), at] = rng.standard_normal(rows)
    got = w.gemm(Tensor.from_data(x).to(device), None, False, True, True).resolve().to(Device.CPU).storage
    want = x[np.arange(rows), at].astype(np.float64)[:, None] * wf[:, at].T
    assert (np.abs(got - want) <= 4 * 2.0**-24 * np.abs(want)).all()


@pytest.mark.parametrize("wt", ["f32", "q8_0f"])
def test_rows_of_four_million(device, wt):
    """Row strides that the limb kernel's 32-bit offsets do not reach: f32 on the f32 kernel, Q8_0F weights on the generic one."""
    n, rows, k = 50, 49, 4_000_000
    gen = torch.Generator("cuda:0").manual_seed(1)
    x = torch.randn((rows, k), generator=gen, device="cuda:0")
    t = lambda v: Tensor(tuple(v.shape), DType.F32, device, v.view(torch.uint8).reshape(-1))
    w = t(torch.randn((n, k), generator=gen, device="cuda:0"))
    if wt == "q8_0f":
        w = Quantizer(Quantization.SInt8).quantize(w)
        codes, scales = w.storage[: n * k].view(torch.int8).view(-1, 32), w.storage[(n * k + 255) // 256 * 256 :].view(torch.float32)[: n * k // 32]
        wf = (codes.float() * scales[:, None]).view(n, k)
    else:
        wf = w.storage.view(torch.float32).view(n, k)
    got = w.gemm(t(x), None, False, True, True).resolve().storage.view(torch.float32)[: rows * n].view(rows, n).double()
    want = torch.zeros((rows, n), dtype=torch.float64, device="cuda:0")
    for lo in range(0, k, 1 << 19):
        want += x[:, lo : lo + (1 << 19)].double() @ wf[:, lo : lo + (1 << 19)].double().T
    # k roundings, each at most 2^-24 of a partial sum of about sqrt(k), of either sign: eight times their root mean square
    assert ((got - want).abs() <= 8 * 2.0**-24 * k).all()


@pytest.mark.parametrize("rows,n,k", [(17, 127, 96), (200, 2560, 10240), (300, 100, 4096), (64, 500, 64)])
def test_codes_with_a_bias_on_the_weight_rows_of_a_row_major_output(device, rows, n, k):
    """W.gemm(x, bias, False, True, False): out [n, rows] with a bias per column, the kernel's row axis, also where K is shared, and with
    an activation behind it."""
    rng = np.random.default_rng(rows + n)
    w = Quantizer(Quantization.SInt8).quantize(Tensor.from_data((rng.standard_normal((n, k)) / math.sqrt(k)).astype(np.float32)).to(device))
    x, bias = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal(rows).astype(np.float32)
    wf = dequantize(w).to(Device.CPU).storage
    t = lambda v: Tensor.from_data(v).to(device)
    want = wf.astype(np.float64) @ x.astype(np.float64).T + bias
    limit = bound(wf, x.T, bias)
    got = w.gemm(t(x), t(bias), False, True, False).resolve().to(Device.CPU).storage
    assert (np.abs(got - want) <= limit).all()
    got = w.gemm(t(x), t(bias), False, True, False).silu().resolve().to(Device.CPU).storage
    # silu's slope is at most 1.1; the hardware's exponential and reciprocal are within 2^-22 of their values for these arguments
    assert (np.abs(got - want / (1 + np.exp(-want))) <= 1.1 * limit + 2.0**-20 * np.abs(want)).all()


def test_a_plan_gives_the_same_bits_whatever_workspace_came_before(device):
    """A plan offers its product first to the family that took it last; a workspace given on one call and not on the next must lead
    where rt_matmul_enqueue_ws leads without a plan."""
    import ctypes

    from ratchet_amd import _ffi

    rng = np.random.default_rng(9)
    L = _ffi.lib()
    dev = lambda v: torch.from_numpy(v).to("cuda:0")
    for n, k, rows in ((384, 1536, 48), (300, 2048, 64), (384, 1536, 200), (384, 384, 48)):
        w, x, bias = (dev(rng.standard_normal(s).astype(np.float32)) for s in ((n, k), (rows, k), (n,)))
        desc = _ffi.make_desc(_ffi.RT_F32, (n, k), _ffi.RT_F32, (rows, k), False, True, True, _ffi.RT_F32, (n,))
        need, plan = ctypes.c_uint64(), ctypes.c_void_p()
        assert L.rt_matmul_workspace_bytes(device.ctx, ctypes.byref(desc), ctypes.byref(need)) == _ffi.RT_OK
        ws = torch.empty(max(need.value, 16), dtype=torch.uint8, device="cuda:0")
        assert L.rt_matmul_plan_create(device.ctx, ctypes.byref(desc), _ffi.RT_ACT_NONE, ctypes.byref(plan)) == _ffi.RT_OK
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        ptrs = (w.data_ptr(), x.data_ptr(), bias.data_ptr())
        try:
            for size in (need.value, 0, 0, need.value, need.value, 0):
                a, b = (torch.full((rows, n), float("nan"), device="cuda:0") for _ in range(2))
                args = (ctypes.c_void_p(ws.data_ptr()) if size else None, size, stream)
                assert L.rt_matmul_plan_enqueue(plan, *ptrs, ctypes.c_void_p(a.data_ptr()), *args) == _ffi.RT_OK
                assert L.rt_matmul_enqueue_ws(device.ctx, ctypes.byref(desc), *ptrs, ctypes.c_void_p(b.data_ptr()), _ffi.RT_ACT_NONE, *args) == _ffi.RT_OK
                assert torch.equal(a, b), (n, k, rows, size)
        finally:
            L.rt_matmul_plan_destroy(plan)
