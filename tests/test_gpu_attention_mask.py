"""Mask tensors in the attention: rows of any alignment (a block ahead through registers), of whole 16-byte vectors (staged), and many query rows
(attention_long_kernel), at the edges of blocks of 64 and 128 keys, with the causal flag beside them, rows without a visible key, and -inf, lowest
and finite values, against float64.

The tolerance: scores are f32 sums of head_dim exact products, probabilities are rounded to f16 (2^-11 of each), sums over the keys are f32 and the
result is rounded to f16 (2^-11)."""
import math

import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F32 if t.dtype == torch.float32 else DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


@pytest.mark.parametrize("mask", [torch.float32, torch.float16])
@pytest.mark.parametrize("heads,head_dim,rows,keys", [
    (2, 40, 3, 3), (3, 64, 17, 63), (2, 96, 65, 65), (2, 128, 130, 127), (3, 80, 70, 257), (2, 72, 100, 191),   # eight wavefronts
    (2, 64, 200, 264), (3, 128, 65, 320),                                                                  # rows of whole vectors
    (2, 80, 70, 1281), (3, 64, 65, 1411), (2, 40, 33, 1407),                                                 # sixteen
    (80, 64, 129, 256), (80, 80, 255, 257), (54, 96, 300, 319), (40, 128, 400, 321), (33, 128, 513, 1027), (20, 96, 1000, 1000),  # many query rows
])
def test_edges(device, heads, head_dim, rows, keys, mask):
    gen = torch.Generator("cuda:0").manual_seed(heads + head_dim + rows + keys)
    q = torch.randn((1, heads, rows, head_dim), generator=gen, device="cuda:0").half()
    k, v = (torch.randn((1, heads, keys, head_dim), generator=gen, device="cuda:0").half() for _ in range(2))
    m = torch.randn((rows, keys), generator=gen, device="cuda:0")
    m[torch.rand((rows, keys), generator=gen, device="cuda:0") < 0.3] = float("-inf")
    m[torch.rand((rows, keys), generator=gen, device="cuda:0") < 0.05] = torch.finfo(mask).min
    m[:, 0] = 0.0
    if rows > 2:
        m[1] = float("-inf")  # no visible key
    m = m.to(mask)
    for causal in (False, True):
        got = tensor(device, q).attention(tensor(device, k), tensor(device, v), tensor(device, m), causal=causal and keys >= rows).resolve()
        got = got.storage.view(torch.float16)[: q.numel()].view(q.shape).double()
        s = q.double() @ k.double().transpose(-1, -2).contiguous() / math.sqrt(head_dim) + m.double()
        if causal and keys >= rows:
            s = s.masked_fill(torch.arange(keys, device="cuda:0")[None, :] > torch.arange(rows, device="cuda:0")[:, None] + (keys - rows), float("-inf"))
        p = torch.softmax(s, -1)
        want, mag = p @ v.double(), p @ v.double().abs()
        seen = torch.ones(rows, dtype=torch.bool, device="cuda:0")
        if rows > 2:
            seen[1] = False
            assert got[:, :, 1].isnan().all()
        err = (got - want).abs()[:, :, seen]
        assert (err <= (2.0**-11 * want.abs() + (2.0**-11 + 2.0**-19) * mag + 2.0**-25)[:, :, seen]).all(), float((err / mag[:, :, seen]).max())
