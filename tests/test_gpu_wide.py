"""The 320 x 256 tiles of the f16 GEMM (gemm_nt_wide_kernel) and the order tiles are dealt to the XCDs in, at the sizes where they can
go wrong, against float64.

The tolerance: a product of K terms rounds its f32 accumulator once per MFMA of 32, each time by at most 2^-24 of the magnitudes
summed, then the bias and the result's rounding to f16 (2^-11)."""
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


def check(device, m, k, n, weight_first):
    gen = torch.Generator("cuda:0").manual_seed(m + k + n)
    w, x, bias = (torch.randn(s, generator=gen, device="cuda:0").half() for s in ((m, k), (n, k), (m,)))
    if weight_first:  # Linear: out [n, m], contiguous along the weight's rows
        got = tensor(device, w).gemm(tensor(device, x), tensor(device, bias), False, True, True).resolve()
    else:  # x . w^T, the operands exchanged inside
        got = tensor(device, x).gemm(tensor(device, w), tensor(device, bias), False, True, False).resolve()
    got = got.storage.view(torch.float16)[: n * m].view(n, m)
    for lo in range(0, n, 512):
        xs = x[lo : lo + 512].double()
        want = xs @ w.double().T + bias.double()
        mag = xs.abs() @ w.double().abs().T + bias.double().abs()
        err = (got[lo : lo + 512].double() - want).abs()
        assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 32 + 3) * mag + 2.0**-25).all(), float((err / mag).max())


@pytest.mark.parametrize("weight_first", [True, False])
@pytest.mark.parametrize("m,k,n", [
    (10240, 320, 2048),   # one tile per compute unit, K steps odd in number
    (10240, 384, 1793),   # the last column tile holds one activation row
    (9921, 448, 2047),    # the last row tile holds one weight row; no 16-byte stores
    (9984, 512, 1990),    # a row tile of 64 rows, ragged columns
    (20480, 320, 2050),   # two rounds
])
def test_edges(device, m, k, n, weight_first):
    check(device, m, k, n, weight_first)


@pytest.mark.parametrize("m,k,n", [
    (2560, 512, 2048),    # 16 x 16 tiles of 160 x 128: four row blocks and eight column blocks per XCD
    (1920, 320, 768),     # 12 x 6
    (480, 320, 2048),     # 3 x 16: the columns dealt to eight XCDs
    (1120, 320, 1024),    # 7 x 8
    (1120, 320, 900),     # 7 x 8, the last column tile ragged
    (1000, 320, 1100),    # 7 x 9: not even
])
def test_tile_orders(device, m, k, n):
    check(device, m, k, n, True)


@pytest.mark.parametrize("m,k,n", [
    (8192, 3072, 200),    # 52 x 2, K shared: no cut fetches less than the plain eighths
    (4160, 320, 1000),    # 26 x 8
    (11008, 320, 1000),   # 69 x 8, a share ends inside a row of tiles
    (4096, 1024, 400),    # 64 x 4 tiles of 64 rows
])
def test_tiles_in_row_order(device, m, k, n):
    check(device, m, k, n, True)
