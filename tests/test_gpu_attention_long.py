"""The attention kernel for many query rows (attention_long_kernel: 128 rows of one head per workgroup, a grid of at least 448 of
them, more than 64 rows and from 256 keys on, no mask tensor) and its neighbours on the other side of those rules, at the sizes where it can go wrong, against float64.

The tolerance: a probability is rounded to f16 (2^-11 of itself, 2^-25 absolute below f16's normal numbers) after scores with the
rounding of an f32 sum of head_dim products, the output once more."""
import math

import pytest
import torch

from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,head_dim,rows,keys,scale", [
    (128, 64, 512, 512, None),     # every workgroup resident, paired
    (112, 80, 500, 500, None),     # the last query block and the last key block ragged
    (56, 96, 1025, 1100, None),    # a query block of one row, an odd number of query blocks
    (448, 128, 65, 1, None),       # one key
    (448, 96, 3, 63, None), (460, 80, 128, 65, None), (257, 64, 129, 128, None),
    (256, 128, 256, 191, None),    # causal: the first rows see no key
    (64, 64, 900, 1283, -0.2), (112, 96, 512, 320, 0.0),
    (9, 80, 6600, 192, None),      # few heads: not whole ones per XCD
])
def test_against_float64(device, heads, head_dim, rows, keys, scale, causal):
    gen = torch.Generator("cuda:0").manual_seed(heads + head_dim + rows + keys)
    cap = keys + 3  # a cache with room: rows past `keys` are never read
    q = torch.randn((1, heads, rows, head_dim), generator=gen, device="cuda:0").half()
    k, v = (torch.randn((1, heads, cap, head_dim), generator=gen, device="cuda:0").half() for _ in range(2))
    q[0, 0, rows // 2] *= 30  # a row whose maximum moves far
    k[:, :, keys:], v[:, :, keys:] = math.nan, math.nan
    node = tensor(device, q).attention(tensor(device, k), tensor(device, v), causal=causal, kv_len=keys, scale=scale)
    node.op.use_workspace = False
    got = node.resolve().storage.view(torch.float16)[: q.numel()].view(q.shape).double()
    s = 1 / math.sqrt(head_dim) if scale is None else scale
    for h in range(0, heads, 16):
        sl = slice(h, min(h + 16, heads))
        qd, kd, vd = q[0, sl].double(), k[0, sl, :keys].double(), v[0, sl, :keys].double()
        scores = torch.matmul(qd, kd.transpose(1, 2).contiguous()) * s
        mag = torch.matmul(qd.abs(), kd.abs().transpose(1, 2).contiguous()) * abs(s)
        if causal:
            hidden = torch.arange(keys, device="cuda:0")[None, :] > torch.arange(rows, device="cuda:0")[:, None] + (keys - rows)
            scores = scores.masked_fill(hidden, -math.inf)
        p = torch.softmax(scores, -1)
        want = torch.matmul(p, vd)
        # a probability's relative error: f16's, and that of its score and of the row's maximum
        e = 2.0**-11 + 2.0**-24 * ((head_dim / 32 + 4) * mag + 8)
        bound = torch.matmul(2 * e.amax(-1, keepdim=True) * p + 2.0**-25, vd.abs()) + 2.0**-11 * want.abs() + 2.0**-25
        g = got[0, sl]
        assert torch.equal(torch.isnan(g), torch.isnan(want))
        ok = ((g - want).abs() <= bound) | torch.isnan(want)
        assert ok.all(), float(((g - want).abs() / bound)[~torch.isnan(want)].max())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,head_dim,rows,keys", [(448, 64, 64, 300), (512, 96, 16, 130), (512, 128, 1, 90), (448, 80, 65, 300)])
def test_few_rows_of_many_heads(device, heads, head_dim, rows, keys, causal):
    """Both sides of the number of rows from which the kernel for many rows takes over."""
    test_against_float64(device, heads, head_dim, rows, keys, None, causal)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,head_dim,rows,keys", [(112, 64, 512, 512), (64, 80, 900, 960), (150, 96, 300, 320), (56, 128, 1000, 1024)])
def test_the_largest_probability_of_a_block_is_exact(device, heads, head_dim, rows, keys, causal):
    """One key of every block of 64 has the weight, their scores within a factor of 2^8 of each other and in any order, and the values
    nearly cancel: a probability relative to its own block's maximum is exactly 1, so what is left is the f32 arithmetic and
    the output's rounding.  Relative to the row's maximum each would be off by up to 2^-11 of itself."""
    gen = torch.Generator("cuda:0").manual_seed(heads + rows)
    q, k = (torch.zeros((1, heads, n, head_dim), dtype=torch.float16, device="cuda:0") for n in (rows, keys))
    v = torch.randn((1, heads, keys, head_dim), generator=gen, device="cuda:0").half()
    q[..., 0] = 1
    k[..., 0] = -300
    at = torch.arange(0, keys, 64, device="cuda:0") + torch.randint(0, 64, (keys // 64,), generator=gen, device="cuda:0")
    k[0, :, at, 0] = torch.rand((heads, len(at)), generator=gen, device="cuda:0").mul(5).sub(2.5).half()
    node = tensor(device, q).attention(tensor(device, k), tensor(device, v), causal=causal, kv_len=keys, scale=1.0)
    node.op.use_workspace = False
    got = node.resolve().storage.view(torch.float16)[: q.numel()].view(q.shape).double()[0]
    s = k[0, :, None, :, 0].double().expand(heads, rows, keys)
    if causal:
        s = s.masked_fill(torch.arange(keys, device="cuda:0")[None, :] > torch.arange(rows, device="cuda:0")[:, None] + (keys - rows), -math.inf)
    p = torch.softmax(s, -1)
    want, mag = torch.matmul(p, v[0].double()), torch.matmul(p, v[0].double().abs())
    # exp2 of a difference of scores of up to 2^3: 2^-21 of itself; a sum over the blocks
    hot = p.amax(-1, keepdim=True) > 1e-3 * (p.sum(-1, keepdim=True))
    seen = (s > -100).any(-1, keepdim=True) & hot
    ok = ((got - want).abs() <= 2.0**-11 * want.abs() + 2.0**-25 + 2.0**-18 * mag) | ~seen
    assert ok.all(), float(((got - want).abs() / mag)[seen.expand_as(want)].max())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,head_dim,rows,keys,scale", [
    (448, 128, 65, 256, None), (460, 80, 128, 257, None), (257, 64, 129, 319, None),
    (150, 128, 350, 256, None),   # causal: the first rows see no key
    (9, 80, 6600, 300, None),     # few heads: not whole ones per XCD
    (448, 96, 66, 1030, -0.2), (230, 64, 200, 700, 0.0), (448, 80, 100, 255, None)])
def test_edges_from_four_key_blocks_on(device, heads, head_dim, rows, keys, scale, causal):
    test_against_float64(device, heads, head_dim, rows, keys, scale, causal)
