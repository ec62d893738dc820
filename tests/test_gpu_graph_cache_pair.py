"""The two cache writes of an attention run in one launch; every other arrangement of them gives the same, bit for bit."""
import pytest
import torch

import ratchet_amd.tensor as mirror
from ratchet_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def tensor(device, t):
    return Tensor(tuple(t.shape), DType.F16, device, t.contiguous().view(torch.uint8).reshape(-1))


def values(t):
    return t.storage.view(torch.float16)[: t.numel()].view(t.shape)


@pytest.mark.parametrize("arrangement", ["together", "keys first", "values first", "one cache for both", "other offsets", "fresh"])
def test_cache_writes_of_an_attention(device, monkeypatch, arrangement):
    H, D, cap, past, new = 3, 64, 40, 17, 5
    gen = torch.Generator("cuda:0").manual_seed(3)
    q, k, v = (torch.randn((1, new, H * D), generator=gen, device="cuda:0").half() for _ in range(3))
    kc, vc = (torch.randn((1, H, cap, D), generator=gen, device="cuda:0").half() for _ in range(2))
    calls = []
    real = mirror._ffi.lib().rt_cache_write_kv_enqueue

    class Counting:
        def __getattr__(self, name):
            f = getattr(mirror._ffi._lib, name)
            if name == "rt_cache_write_kv_enqueue":
                return lambda *a: (calls.append(1), real(*a))[1]
            return f

    counting = Counting()
    monkeypatch.setattr(mirror._ffi, "lib", lambda: counting)
    KC, VC = tensor(device, kc.clone()), tensor(device, vc.clone())
    if arrangement == "one cache for both":
        VC = KC
    voff = past + 3 if arrangement == "other offsets" else past
    if arrangement == "fresh":
        keys, vals = KC.cache(tensor(device, k.view(1, new, H, D).transpose(1, 2)), 2, past), VC.cache(tensor(device, v.view(1, new, H, D).transpose(1, 2)), 2, past)
    else:
        keys, vals = KC.cache_write(tensor(device, k), past), VC.cache_write(tensor(device, v), voff)
    if arrangement == "keys first":
        keys.resolve()
    if arrangement == "values first":
        vals.resolve()
    kv_len = past + new
    got = values(tensor(device, q).attention(keys, vals, causal=True, kv_len=kv_len, merge_heads=True).resolve())
    assert len(calls) == (1 if arrangement == "together" else 0)
    heads = lambda t: t.view(1, new, H, D).transpose(1, 2)
    kd, vd = kc.clone(), vc.clone()
    kd[:, :, past:kv_len] = heads(k)
    if arrangement == "one cache for both":
        kd[:, :, past:kv_len] = heads(v)
        vd = kd
    else:
        vd[:, :, voff : voff + new] = heads(v)
    want = values(tensor(device, q.view(1, new, H, D).transpose(1, 2)).attention(tensor(device, kd[:, :, :kv_len]), tensor(device, vd[:, :, :kv_len]), causal=True).resolve())
    assert torch.equal(got, want.transpose(1, 2).reshape(1, new, H * D))
    if arrangement != "fresh":
        assert torch.equal(values(KC), kd) and torch.equal(values(VC), vd)


@pytest.mark.parametrize("reader", ["queries", "values"])
def test_what_reads_the_caches_between_the_writes(device, reader):
    """Queries from an attention over the same caches run before the writes, and values made of the key cache behind the keys' write."""
    H, D, n = 2, 64, 16
    gen = torch.Generator("cuda:0").manual_seed(5)
    q, k1, v1, k2, v2, k0, v0 = (torch.randn((1, H, n, D), generator=gen, device="cuda:0").half() for _ in range(7))
    KC, VC = tensor(device, k0.clone()), tensor(device, v0.clone())

    def attend(first, lazy):
        step = (lambda t: t) if lazy else (lambda t: t.resolve())
        q2, keys, vals = tensor(device, q), tensor(device, k2), tensor(device, v2)
        if reader == "queries":
            q2 = step(first.attention(step(KC.cache_write(tensor(device, k1), 0)), step(VC.cache_write(tensor(device, v1), 0))))
        written = step(KC.cache_write(keys, 0))
        if reader == "values":
            vals = step(KC.gelu())
        return values(q2.attention(written, step(VC.cache_write(vals, 0))).resolve()).clone()

    want = attend(tensor(device, q), lazy=False)
    values(KC).copy_(k0), values(VC).copy_(v0)
    assert torch.equal(attend(tensor(device, q), lazy=True), want)


@pytest.mark.parametrize("reader", ["values are the key cache", "keys are the value cache", "keys are a write into the value cache", "values are a write into the keys",
                                    "one memory for both"])
def test_writes_whose_order_matters(device, reader):
    """One cache is the other's source, or both are one memory in two tensors: as one write after the other leaves it."""
    H, D, n = 4, 64, 256
    gen = torch.Generator("cuda:0").manual_seed(9)
    q, k, v, x, kc, vc = (torch.randn((1, H, n, D), generator=gen, device="cuda:0").half() for _ in range(6))

    def attend(lazy):
        step = (lambda t: t) if lazy else (lambda t: t.resolve())
        memory = kc.clone()
        KC, VC = tensor(device, memory), tensor(device, memory if reader == "one memory for both" else vc.clone())
        keys, vals = tensor(device, k.clone()), tensor(device, v)
        if reader == "values are the key cache":
            vals = KC
        if reader == "keys are the value cache":
            keys = VC
        if reader == "keys are a write into the value cache":
            keys = step(VC.cache_write(tensor(device, x), 0))
        written = step(KC.cache_write(keys, 0))
        if reader == "values are a write into the keys":
            vals = step(keys.cache_write(tensor(device, x), 0))
        out = tensor(device, q).attention(written, step(VC.cache_write(vals, 0))).resolve()
        return [values(t).clone() for t in (out, KC, VC)]

    assert all(torch.equal(a, b) for a, b in zip(attend(lazy=True), attend(lazy=False)))
