"""The two cache writes of an attention share a launch only where their order cannot matter.  A library that writes host memory, a
value row before each key row as the two halves of a launch may, stands in for the device: what comes out is what one write
after the other leaves."""
import ctypes

import pytest
import torch

import ratchet_amd.tensor as mirror
from ratchet_amd import Device, DType, Tensor

H, CAP, D = 2, 4, 8


class HostLibrary:
    """rt_cache_write_enqueue and rt_cache_write_kv_enqueue for [1, H, CAP, D] f16 caches in host memory."""

    def __init__(self):
        self.pairs = 0

    @staticmethod
    def write(cache, src, strides, heads, capacity, offset, rows, head_dim):
        for r in range(rows):
            for h in range(heads):
                yield lambda r=r, h=h: ctypes.memmove(cache + 2 * head_dim * (h * capacity + offset + r), src + 2 * (h * strides[1] + r * strides[2]), 2 * head_dim)

    def rt_cache_write_enqueue(self, ctx, dt, cache, src, strides, dst, batch, heads, capacity, offset, rows, head_dim, stream):
        for step in self.write(cache, src, strides, heads, capacity, offset, rows, head_dim):
            step()
        return 0

    def rt_cache_write_kv_enqueue(self, ctx, dt, kc, ks, vc, vs, strides, batch, heads, capacity, offset, rows, head_dim, stream):
        self.pairs += 1
        for a, b in zip(*(self.write(c, s, strides, heads, capacity, offset, rows, head_dim) for c, s in ((vc, vs), (kc, ks)))):
            a(), b()
        return 0


def arrange(name, tensor):
    """The keys' and the values' write, and the memory that both leave behind."""
    gen = torch.Generator().manual_seed(7)
    new = lambda rows=CAP: torch.randn((1, H, rows, D), generator=gen).half()
    kc, vc, k, v, x = new(), new(), new(), new(), new()
    KC, VC = tensor(kc), tensor(vc)
    keys, values = tensor(k), tensor(v)
    if name == "values are the key cache":
        values = KC
    if name == "values are the key cache in another tensor":
        values = tensor(kc)
    if name == "keys are the value cache":
        keys = VC
    if name == "keys are a write into the value cache":
        keys = VC.cache_write(tensor(x), 0)
    if name == "values are a write into the keys":
        values = keys.cache_write(tensor(x), 0)
    if name == "keys are the values that are written":
        values = tensor(v)
        written = VC.cache_write(values, 0)
        return KC.cache_write(written.cache_write(tensor(x), 0), 0), written, (kc, vc, k, v)
    if name == "one memory for both":
        VC, vc = tensor(kc), kc
    if name == "memories that overlap":
        both = torch.randn((H * CAP * D + 2 * D,), generator=gen).half()
        kc, vc = both[: H * CAP * D].view(1, H, CAP, D), both[2 * D :].view(1, H, CAP, D)
        KC, VC = tensor(kc), tensor(vc)
    return KC.cache_write(keys, 0), VC.cache_write(values, 0), (kc, vc, k, v)


@pytest.mark.parametrize("name", ["apart", "values are the key cache", "values are the key cache in another tensor", "keys are the value cache",
                                  "keys are a write into the value cache", "values are a write into the keys", "keys are the values that are written",
                                  "one memory for both", "memories that overlap"])
def test_order_of_the_writes(monkeypatch, name):
    device = Device("gpu")
    device._ctx = object()
    library = HostLibrary()
    monkeypatch.setattr(mirror._ffi, "lib", lambda: library)
    tensor = lambda t: Tensor(tuple(t.shape), DType.F16, device, t.view(torch.uint8).reshape(-1))
    left = []
    for pair in (False, True):
        k, v, memory = arrange(name, tensor)
        if pair:
            mirror._write_key_and_value(k, v, 0)
        for t in (k, v):
            if t.storage is None:
                t._execute(0)
        left.append([m.clone() for m in memory])
    assert library.pairs == (name == "apart")
    assert all(torch.equal(a, b) for a, b in zip(*left))
