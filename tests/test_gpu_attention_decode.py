"""One query row (a decode step): the kernels that take it in one launch (128, 256, 448 keys) and split over workgroups, with and without a
mask tensor, and the merge of split launches with several query rows, against float64.

The tolerance: scores are f32 sums of head_dim exact products (2^-24 of the magnitudes, 8 roundings at the most), probabilities and the sums
over the keys are f32; the tiled kernels round probabilities to f16 (2^-11 of each); the result is rounded to f16 (2^-11)."""
import math

import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F32 if t.dtype == torch.float32 else DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


def check(device, heads, head_dim, rows, keys, mask=None, causal=False, capacity=None, batch=1, probability=2.0**-20):
    gen = torch.Generator("cuda:0").manual_seed(heads + head_dim + rows + keys)
    cap = capacity or keys
    q = torch.randn((batch, heads, rows, head_dim), generator=gen, device="cuda:0").half()
    k, v = (torch.randn((batch, heads, cap, head_dim), generator=gen, device="cuda:0").half() for _ in range(2))
    k[:, :, keys:], v[:, :, keys:] = float("nan"), float("nan")  # rows of the cache past the keys are never used
    m = None
    if mask is not None:
        m = torch.randn((rows, keys), generator=gen, device="cuda:0")
        m[torch.rand((rows, keys), generator=gen, device="cuda:0") < 0.3] = float("-inf")
        m[:, keys // 2] = 0.0
        m = m.to(mask)
    out = tensor(device, q).attention(tensor(device, k), tensor(device, v), tensor(device, m) if m is not None else None, causal=causal, kv_len=keys).resolve()
    got = out.storage.view(torch.float16)[: q.numel()].view(q.shape).double()
    kd, vd = k[:, :, :keys].double(), v[:, :, :keys].double()
    s = q.double() @ kd.transpose(-1, -2).contiguous() / math.sqrt(head_dim)
    if m is not None:
        s = s + m.double()
    if causal:
        s = s.masked_fill(torch.arange(keys, device="cuda:0")[None, :] > torch.arange(rows, device="cuda:0")[:, None] + (keys - rows), float("-inf"))
    p = torch.softmax(s, -1)
    want, mag = p @ vd, p @ vd.abs()
    # a score's error moves its probability by as much: magnitudes up to 6 head_dim / sqrt(head_dim), times log2(e) and exp2's own error
    assert ((got - want).abs() <= 2.0**-11 * want.abs() + (probability + 2.0**-19) * mag + 2.0**-25).all(), float(((got - want).abs() / mag).max())


@pytest.mark.parametrize("mask", [None, torch.float32, torch.float16])
@pytest.mark.parametrize("heads,head_dim,keys", [
    (3, 64, 1), (5, 40, 2), (2, 128, 16), (8, 80, 127), (32, 96, 128),          # one launch, 256 threads
    (4, 80, 129), (7, 8, 200), (2, 128, 256),                                  # 512
    (4, 80, 257), (3, 64, 447), (2, 128, 448),                                 # 1024
    (4, 80, 449), (2, 128, 513), (3, 40, 1331), (2, 64, 4097),                 # two launches
])
def test_one_row(device, heads, head_dim, keys, mask):
    check(device, heads, head_dim, 1, keys, mask)
    check(device, heads, head_dim, 1, keys, mask, causal=True, capacity=keys + 37, batch=2)


def test_no_visible_key(device):
    for keys in (5, 200, 300, 700):
        q, k, v = (tensor(device, torch.randn(s, device="cuda:0").half()) for s in ((1, 2, 1, 64), (1, 2, keys, 64), (1, 2, keys, 64)))
        m = torch.full((1, keys), float("-inf"), device="cuda:0")
        out = q.attention(k, v, tensor(device, m)).resolve()
        assert out.storage.view(torch.float16)[:128].isnan().all()
        m[0, keys - 1] = 0.0  # ... and one: its value, exactly
        out = q.attention(k, v, tensor(device, m)).resolve()
        assert torch.equal(out.storage.view(torch.float16)[:128].view(2, 64), v.storage.view(torch.float16)[: 2 * keys * 64].view(2, keys, 64)[:, -1])


@pytest.mark.parametrize("heads,head_dim,rows,keys", [
    (8, 80, 400, 400), (6, 40, 332, 332), (2, 128, 64, 1024), (1, 8, 1, 4096), (3, 72, 65, 700), (1, 96, 2, 2048), (5, 64, 129, 1000), (20, 80, 70, 390),
])
def test_merge_of_split_launches(device, heads, head_dim, rows, keys):
    check(device, heads, head_dim, rows, keys, probability=2.0**-11)
    check(device, heads, head_dim, rows, keys, causal=True, probability=2.0**-11)


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("keys", [1, 64, 100, 200, 256, 300, 448, 449, 512, 576, 700])
def test_infinite_value_at_the_last_key(device, keys, masked):
    """What the kernels read in place of keys past the last one leaves no NaN: an infinite value stays infinite."""
    gen = torch.Generator("cuda:0").manual_seed(keys)
    q = torch.randn((1, 2, 1, 64), generator=gen, device="cuda:0").half()
    k, v = (torch.randn((1, 2, keys, 64), generator=gen, device="cuda:0").half() for _ in range(2))
    v[:, :, -1, 3], v[:, :, -1, 60] = float("inf"), float("-inf")
    mask = tensor(device, torch.zeros((1, keys), device="cuda:0")) if masked else None
    got = tensor(device, q).attention(tensor(device, k), tensor(device, v), mask).resolve().storage.view(torch.float16)[:128].view(2, 64)
    assert (got[:, 3] == float("inf")).all() and (got[:, 60] == float("-inf")).all()
    finite = torch.ones(64, dtype=torch.bool, device="cuda:0")
    finite[3] = finite[60] = False
    assert got[:, finite].isfinite().all()


@pytest.mark.parametrize("stride", [0, 8])
@pytest.mark.parametrize("keys", [100, 300, 700])
def test_infinite_value_where_rows_share_memory(device, keys, stride):
    """Rows of values that begin less than a row apart: a row past the last key would lie inside the values, and leaves no NaN either."""
    gen = torch.Generator("cuda:0").manual_seed(keys)
    q, k, v = (torch.randn(s, generator=gen, device="cuda:0").half() for s in ((1, 2, 1, 64), (1, 2, keys, 64), (1, 2, keys, 64)))
    last = (keys - 1) * stride + 63
    v.view(2, -1)[:, last] = float("inf")
    node = tensor(device, q).attention(tensor(device, k), tensor(device, v), None)
    node.op.desc.v_strides[2] = stride
    got = node.resolve().storage.view(torch.float16)[:128].view(2, 64)
    rows = v.as_strided((2, keys, 64), (keys * 64, stride, 1)).double()
    p = torch.softmax((k[0].double() @ q[0].double().transpose(1, 2).contiguous()).transpose(1, 2) / 8, -1)
    assert (got[:, 63] == float("inf")).all()
    want, mag = ((p[:, 0, :, None] * r).sum(1) for r in (rows[..., :63], rows[..., :63].abs()))
    assert ((got[:, :63].double() - want).abs() <= 2.0**-11 * want.abs() + (2.0**-20 + 2.0**-19) * mag + 2.0**-25).all()
