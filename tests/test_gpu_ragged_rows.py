"""Attention operator by operator over lengths that are no multiple of eight, and softmax rows that start and end anywhere, against float64.

Tolerances: products of f16 numbers are exact in the MFMA, whose f32 accumulator rounds once per 32 k by 2^-24 of the magnitudes summed at the
most, then the result is rounded to f16 (2^-11).  Softmax as in test_gpu_softmax_rows."""
import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F32 if t.dtype == torch.float32 else DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


def values(t):
    return t.storage.view(torch.float16)[: t.numel()].view(t.shape).double()


def close(got, want, mag, k):
    err = (got - want).abs()
    assert (err <= 2.0**-11 * want.abs() + 2.0**-24 * (k / 32 + 3) * mag + 2.0**-25).all(), float((err / mag.clamp(min=1e-30)).max())


@pytest.mark.parametrize("head_dim", [8, 64, 80, 96, 128])
@pytest.mark.parametrize("heads,rows,keys", [(3, 64, 9), (2, 65, 15), (5, 71, 66), (1, 100, 127), (6, 129, 129), (2, 254, 254), (8, 130, 401), (3, 964, 964), (1, 200, 1027), (2, 64, 64)])
def test_probabilities_times_values(device, heads, rows, keys, head_dim):
    gen = torch.Generator("cuda:0").manual_seed(heads + rows + keys + head_dim)
    p = torch.randn((heads, rows, keys), generator=gen, device="cuda:0").half()
    v = torch.randn((heads, keys, head_dim), generator=gen, device="cuda:0").half()
    got = values(tensor(device, p).matmul(tensor(device, v), False, False).resolve())
    close(got, p.double() @ v.double(), p.double().abs() @ v.double().abs(), keys)


@pytest.mark.parametrize("heads,rows,keys,head_dim", [(2, 65, k, n) for k, n in ((31, 48), (33, 48), (63, 56), (65, 96), (127, 104), (129, 128))] +
                         [(32, 577, k, n) for k, n in ((95, 56), (97, 96), (159, 48), (161, 40), (159, 104), (161, 128))])
def test_probabilities_times_values_on_both_sides_of_the_rule(device, heads, rows, keys, head_dim):
    test_probabilities_times_values(device, heads, rows, keys, head_dim)


@pytest.mark.parametrize("head_dim", [8, 40, 64, 96, 128, 200])
@pytest.mark.parametrize("heads,rows,keys", [(3, 64, 161), (2, 65, 162), (5, 130, 167), (1, 200, 254), (6, 300, 301), (2, 964, 964), (2, 1027, 333)])
def test_scores(device, heads, rows, keys, head_dim):
    gen = torch.Generator("cuda:0").manual_seed(heads + rows + keys + head_dim)
    q, k = (torch.randn((heads, n, head_dim), generator=gen, device="cuda:0").half() for n in (rows, keys))
    got = values(tensor(device, q).matmul(tensor(device, k), False, True).resolve())
    kt = k.double().transpose(1, 2).contiguous()
    close(got, q.double() @ kt, q.double().abs() @ kt.abs(), head_dim)


@pytest.mark.parametrize("n", [1000, 1001, 853, 51])  # a vocabulary of any size: rows of the output that start on 16, 2, 2 and 2 bytes
@pytest.mark.parametrize("rows,k", [(300, 512), (70, 288), (600, 1056)])
def test_linear_outputs_of_any_width(device, rows, n, k):
    gen = torch.Generator("cuda:0").manual_seed(rows + n + k)
    w, x, b = (torch.randn(s, generator=gen, device="cuda:0").half() for s in ((n, k), (rows, k), (n,)))
    got = values(tensor(device, w).gemm(tensor(device, x), tensor(device, b), False, True, True).resolve())
    wt = w.double().T.contiguous()
    close(got, x.double() @ wt + b.double(), x.double().abs() @ wt.abs() + b.double().abs(), k)


@pytest.mark.parametrize("dt,n", [("f32", 1), ("f32", 3), ("f32", 5), ("f32", 250), ("f32", 255), ("f32", 257), ("f32", 874), ("f32", 1025), ("f32", 2045), ("f32", 2049),
                                  ("f16", 1), ("f16", 7), ("f16", 9), ("f16", 254), ("f16", 505), ("f16", 513), ("f16", 964), ("f16", 1027), ("f16", 2049), ("f16", 4082), ("f16", 4091)])
def test_softmax_rows_that_start_anywhere(device, dt, n):
    softmax_rows(device, dt, 203, n)


@pytest.mark.parametrize("dt,n", [("f32", 129), ("f32", 250), ("f32", 257), ("f32", 1025), ("f32", 2045), ("f16", 129), ("f16", 254), ("f16", 505), ("f16", 1027), ("f16", 2049), ("f16", 4082)])
@pytest.mark.parametrize("rows", [1025, 3001])  # many of them: a wavefront a row (fewer: a workgroup)
def test_many_softmax_rows_that_start_anywhere(device, dt, rows, n):
    softmax_rows(device, dt, rows, n)


def softmax_rows(device, dt, rows, n):
    t, d = (torch.float32, DType.F32) if dt == "f32" else (torch.float16, DType.F16)
    x = (torch.randn((rows, n), generator=torch.Generator("cuda:0").manual_seed(n), device="cuda:0") * 3).to(t)
    x[4], x[5, n - 1], x[6, 0] = -float("inf"), float("nan"), float("inf")  # none of it reaches a neighbour's row
    e = torch.exp(x.double() - x.double().amax(-1, keepdim=True))
    want = e / e.sum(-1, keepdim=True)
    got = Tensor((rows, n), d, device, x.clone().view(torch.uint8).reshape(-1)).softmax(1).resolve().storage.view(t)[: x.numel()].view(x.shape).double()
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.isnan(want[4:7]).all()
    size = (x.double() - x.double().amax(-1, keepdim=True)).abs().clamp(max=200)
    rel = 2.0**-24 * (size + 4 + 2 + 32 + 6 + 1) + (2.0**-11 if dt == "f16" else 0)
    tiny = 2.0**-25 if dt == "f16" else 2.0**-149 * 2
    ok = ((got - want).abs() <= rel * want + tiny) | torch.isnan(want)
    assert ok.all(), float(((got - want).abs() / want.clamp(min=1e-38))[~torch.isnan(want)].max())
