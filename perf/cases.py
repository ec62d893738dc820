"""What a program built on this library has it do, as cases that can be timed and compared.

The library is the matrix-product path of a transformer runtime: linear layers over f32, f16, Q8_0 and Q4_K weights,
the attention products and the fused attention, activations in the products' epilogues and the key/value cache.  A
case is one pass of such a piece of a model.  Passes go through the C interface of include/ratchet_hip.h the way a
runtime drives it (a plan per product kept from load time, a workspace of the size the library asks for, one enqueue
per operator and pass), except the `nn` cases, which go through the Python modules of ratchet_amd.nn.

Shapes: the Phi-2 (width 2560, inner width 10240, 32 heads of 80) and Phi-3-mini (3072, 8192) layers and the
Whisper-tiny encoder (1500 positions, width 384, 6 heads of 64) that this repository's tests and benchmark use;
`draw` spreads sizes around them.  Activations are N(0, 1), weights N(0, 1/sqrt(K)) and quantized where the case says
so, as a checkpoint's would be.

  linear     one product x.W^T + bias: rows activation rows (1: a decode step; tens: a short prompt; up to a few thousand:
             prefill), n outputs, k inputs, wt the weights' type.  Activations are f16 against f16, Q8_0H and Q4_K weights,
             f32 against f32 and Q8_0F weights.
  mlp        two products, the first with GELU in its epilogue.
  layer      layers decoder layers one after the other: projection to q, k and v in one product, both cache writes,
             causal attention over past + rows cached positions, output projection, and an MLP beside it.
             rows = 1 is a decode step, more a prompt.
  nn         the attention block and the MLP behind it through ratchet_amd.nn, resolved once.
  attention  the fused attention on its own: no mask, the causal flag, or the mask as a tensor.
  scores     attention operator by operator, as the reference's modules spell it: Q.K^T, softmax, P.V.
"""
import ctypes
import math

import torch

import ratchet_amd as ra
from ratchet_amd import _ffi

ACT = {"none": _ffi.RT_ACT_NONE, "gelu": _ffi.RT_ACT_GELU, "silu": _ffi.RT_ACT_SILU}
DT = {"f32": ra.DType.F32, "f16": ra.DType.F16, "q8_0f": ra.DType.Q8_0F, "q8_0h": ra.DType.Q8_0H, "q4_k": ra.DType.Q4_K}
BLOCK = {"f32": 32, "f16": 32, "q8_0f": 32, "q8_0h": 32, "q4_k": 256}
BITS = {"f32": 32, "f16": 16, "q8_0f": 9, "q8_0h": 8.5, "q4_k": 4.5}  # stored per weight
GPU = "cuda:0"

# What a drawn case may cost: the largest listed case of its arithmetic (f32 products run at a sixteenth of the f16 rate).
MOST_FLOPS = {"f16": 2.1e11, "f32": 3.1e10}


def listed():
    return [
        # the smallest call: one decode step's up-projection, Q8_0 weights; latency and one pass over 28 MB
        {"name": "linear_q8h_1", "kind": "linear", "wt": "q8_0h", "rows": 1, "n": 10240, "k": 2560, "act": "none"},
        # token generation: one token through four Phi-2 layers with 1024 cached positions
        {"name": "decode_q8h", "kind": "layer", "wt": "q8_0h", "layers": 4, "rows": 1, "past": 1023, "heads": 32, "head_dim": 80},
        # the same step for a program that builds the lazy graph in Python and resolves it
        {"name": "nn_decode_q8h", "kind": "nn", "wt": "q8_0h", "rows": 1, "past": 1023, "heads": 32, "head_dim": 80},
        # a 512-token prompt through a quantized layer
        {"name": "prefill_q8h", "kind": "layer", "wt": "q8_0h", "layers": 1, "rows": 512, "past": 0, "heads": 32, "head_dim": 80},
        # a long prompt (or a batch of prompts) through an unquantized MLP: the largest product
        {"name": "mlp_f16_2048", "kind": "mlp", "wt": "f16", "rows": 2048, "k": 2560, "n": 10240},
        # Q4_K weights, one token and a prompt of no particular length
        {"name": "mlp_q4k_1", "kind": "mlp", "wt": "q4_k", "rows": 1, "k": 3072, "n": 8192},
        {"name": "mlp_q4k_1000", "kind": "mlp", "wt": "q4_k", "rows": 1000, "k": 3072, "n": 8192},
        # the encoder's MLP in f32: every position of the audio window
        {"name": "mlp_f32_1500", "kind": "mlp", "wt": "f32", "rows": 1500, "k": 384, "n": 1536},
        # weights from this library's quantizer (f32 scales) against f32 activations, a ragged prompt
        {"name": "mlp_q8f_200", "kind": "mlp", "wt": "q8_0f", "rows": 200, "k": 2560, "n": 10240},
        # causal attention over a long prompt
        {"name": "attention_2048", "kind": "attention", "heads": 32, "head_dim": 96, "rows": 2048, "keys": 2048, "mask": "causal"},
        # the encoder's attention as three operators in f32; the row length is no multiple of a cache line
        {"name": "scores_f32_1500", "kind": "scores", "dt": "f32", "heads": 6, "head_dim": 64, "rows": 1500, "keys": 1500},
        # the decoder's attention as three operators in f16
        {"name": "scores_f16_512", "kind": "scores", "dt": "f16", "heads": 32, "head_dim": 80, "rows": 512, "keys": 512},
    ]


def draw(rng):
    def spread(lo, hi, step=1):
        return max(1, round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step

    while True:
        kind = rng.choice(["linear", "linear", "mlp", "mlp", "layer", "nn", "attention", "attention", "scores"])
        if kind in ("linear", "mlp"):
            wt = rng.choice(list(DT))
            k = spread(256, 4096, BLOCK[wt])
            if kind == "linear":
                # a vocabulary may have any number of entries
                n = spread(256, 51865) if rng.random() < 0.3 else spread(256, 16384, 32)
                case = {"kind": kind, "wt": wt, "rows": spread(1, 2048), "n": n, "k": k, "act": rng.choice(list(ACT))}
            else:
                case = {"kind": kind, "wt": wt, "rows": spread(1, 2048), "k": k, "n": rng.choice([8 * k // 3 // BLOCK[wt] * BLOCK[wt], 4 * k])}
        elif kind in ("layer", "nn"):
            wt = rng.choice(["f16", "q8_0h", "q4_k"])
            heads, head_dim = rng.choice([(8, 64), (16, 64), (32, 64), (32, 80), (32, 96), (32, 128)])
            rows, past = rng.choice([(1, spread(16, 4095)), (spread(2, 1024), 0)])
            case = {"kind": kind, "wt": wt, "rows": rows, "past": past, "heads": heads, "head_dim": head_dim}
            if kind == "layer":
                case["layers"] = 4 if rows == 1 else 1
        elif kind == "attention":
            rows = rng.choice([1, spread(2, 2048), spread(128, 2048)])
            case = {"kind": kind, "heads": rng.choice([6, 8, 16, 32, 40]), "head_dim": rng.choice([40, 64, 80, 96, 128]), "rows": rows,
                    "keys": rng.choice([rows, rows + spread(1, 2048)]) if rows > 1 else spread(64, 8192),
                    "mask": rng.choice(["none", "causal", "causal", "f32", "f16"])}
        else:
            rows = spread(16, 1536)
            case = {"kind": kind, "dt": rng.choice(["f16", "f32"]), "heads": rng.choice([6, 8, 16, 32]), "head_dim": rng.choice([64, 80, 96]),
                    "rows": rows, "keys": rows}
        w, f32 = work(case), case.get("wt") in ("f32", "q8_0f") or case.get("dt") == "f32"
        if w["flops"] <= MOST_FLOPS["f32" if f32 else "f16"]:
            return case


# ---- inputs ---------------------------------------------------------------------------------------------------------


def activation_type(wt):
    return "f32" if wt in ("f32", "q8_0f") else "f16"


def torch_type(dt):
    return torch.float32 if dt == "f32" else torch.float16


def normal(gen, shape, dt):
    return torch.randn(shape, generator=gen, device=GPU, dtype=torch.float32).to(torch_type(dt))


def pad256(t):
    return torch.nn.functional.pad(t, (0, -t.numel() % 256))


def weight(gen, n, k, wt, scale=1.0):
    """An n x k weight in the library's storage for `wt`, as bytes."""
    w = torch.randn((n, k), generator=gen, device=GPU, dtype=torch.float32).mul_(scale / math.sqrt(k))
    if wt in ("f32", "f16"):
        return w.to(torch_type(wt)).view(torch.uint8).reshape(-1)
    if wt in ("q8_0f", "q8_0h"):  # one absmax scale per 32 weights: codes, then scales, each padded to 256 bytes
        w = w.view(-1, 32)
        d = w.abs().amax(1).div_(127.0).to(torch.float16 if wt == "q8_0h" else torch.float32)
        q = w.div_(d.float().clamp_(min=1e-30)[:, None]).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([pad256(q.view(torch.uint8).reshape(-1)), pad256(d.view(torch.uint8).reshape(-1))])
    # Q4_K: 256 weights as {f16 d, f16 dmin, 8 six-bit scales and mins in 12 bytes, 128 bytes of nibbles}
    w = w.view(-1, 8, 32)
    low = w.amin(2).clamp_(max=0.0).neg_()
    span = (w.amax(2) + low).div_(15.0)
    d, dmin = span.amax(1).div_(63.0).half(), low.amax(1).div_(63.0).half()
    sc = (span / d.float()[:, None]).round_().clamp_(1, 63)
    mn = (low / dmin.float()[:, None]).round_().clamp_(0, 63)
    q = w.add_((dmin.float()[:, None] * mn)[:, :, None]).div_((d.float()[:, None] * sc)[:, :, None]).round_().clamp_(0, 15)
    sc, mn, q = sc.to(torch.uint8), mn.to(torch.uint8), q.to(torch.uint8)
    head = torch.cat([d[:, None].view(torch.uint8), dmin[:, None].view(torch.uint8),
                      sc[:, :4] | (sc[:, 4:] >> 4 << 6), mn[:, :4] | (mn[:, 4:] >> 4 << 6), (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)], 1)
    return torch.cat([head, (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(-1, 128)], 1).reshape(-1)


_device = None


def device():
    """The library's context: one for the program's life."""
    global _device
    if _device is None:
        _device = ra.Device.request_device(ra.DeviceRequest.GPU)
    return _device


def check(status):
    if status != _ffi.RT_OK:
        raise RuntimeError(ra.lib().rt_last_error(device().ctx).decode() or _ffi.status_string(status))


def ptr(t):
    return None if t is None else t.data_ptr()


class Product:
    """A product compiled once: its plan, the workspace it asks for, its operands and its output."""

    def __init__(self, lhs, lhs_dt, lhs_shape, rhs, rhs_dt, rhs_shape, bias=None, act="none", trans_rhs=False, trans_out=False):
        L, plan, need = ra.lib(), ctypes.c_void_p(), ctypes.c_uint64()
        bias_dt = None if bias is None else DT["f32" if bias.dtype == torch.float32 else "f16"]
        desc = _ffi.make_desc(DT[lhs_dt], lhs_shape, DT[rhs_dt], rhs_shape, False, trans_rhs, trans_out, bias_dt, None if bias is None else bias.shape)
        shape, rank, dt = (ctypes.c_int64 * _ffi.RT_MAX_RANK)(), ctypes.c_int32(), ctypes.c_int32()
        check(L.rt_matmul_infer(ctypes.byref(desc), shape, ctypes.byref(rank), ctypes.byref(dt)))
        check(L.rt_matmul_plan_create(device().ctx, ctypes.byref(desc), ACT[act], ctypes.byref(plan)))
        self.plan, self.destroy = plan, L.rt_matmul_plan_destroy
        check(L.rt_matmul_workspace_bytes(device().ctx, ctypes.byref(desc), ctypes.byref(need)))
        self.workspace = torch.empty(need.value, dtype=torch.uint8, device=GPU) if need.value else None
        self.out = torch.empty(list(shape[:rank.value]), dtype=torch_type("f32" if dt.value == _ffi.RT_F32 else "f16"), device=GPU)
        self.operands = (lhs, rhs, bias)
        self.call = (L.rt_matmul_plan_enqueue, (plan, ptr(lhs), ptr(rhs), ptr(bias), ptr(self.out), ptr(self.workspace), need.value))

    def __del__(self):
        self.destroy(self.plan)


def linear(gen, x, wt, n, act="none", scale=1.0):
    """x [rows, k] . W [n, k]^T + bias, the reference's Linear: W.gemm(x, bias, false, true, true)."""
    rows, k = x.shape
    return Product(weight(gen, n, k, wt, scale), wt, (n, k), x, activation_type(wt), (rows, k), normal(gen, (n,), activation_type(wt)) * 0.02, act,
                   trans_rhs=True, trans_out=True)


def attention_desc(heads, head_dim, rows, keys, q_strides, kv_strides, causal, mask=None):
    d = _ffi.AttentionDesc()
    d.dtype, d.batch, d.heads, d.q_len, d.kv_len, d.head_dim = _ffi.RT_F16, 1, heads, rows, keys, head_dim
    d.q_strides[:], d.k_strides[:], d.v_strides[:] = q_strides, kv_strides, kv_strides
    d.o_strides[:] = [rows * heads * head_dim, head_dim, heads * head_dim]  # [rows, heads * head_dim]
    d.scale, d.causal = 1 / math.sqrt(head_dim), int(causal)
    d.mask_dtype = _ffi.RT_F32 if mask is None or mask.dtype == torch.float32 else _ffi.RT_F16
    d.mask_row_stride = keys
    return d


def attention_call(desc, q, k, v, mask, out):
    """The call, and the tensors it needs alive."""
    need = ctypes.c_uint64()
    check(ra.lib().rt_attention_workspace_bytes(ctypes.byref(desc), ctypes.byref(need)))
    ws = torch.empty(need.value, dtype=torch.uint8, device=GPU) if need.value else None
    args = (device().ctx, ctypes.byref(desc), q if isinstance(q, int) else ptr(q), ptr(k), ptr(v), ptr(mask), ptr(out), ptr(ws), need.value)
    return (ra.lib().rt_attention_enqueue, args), (desc, q, k, v, mask, out, ws)


def tensor(t, shape, dt):
    return ra.Tensor(shape, DT[dt], device(), t.view(torch.uint8).reshape(-1))


def prepare(case, seed):
    gen = torch.Generator(GPU)
    gen.manual_seed(seed)
    kind, calls, keep, out = case["kind"], [], [], []
    if kind == "linear":
        p = linear(gen, normal(gen, (case["rows"], case["k"]), activation_type(case["wt"])), case["wt"], case["n"], case["act"])
        calls, keep, out = [p.call], [p], [p.out]
    elif kind == "mlp":
        up = linear(gen, normal(gen, (case["rows"], case["k"]), activation_type(case["wt"])), case["wt"], case["n"], "gelu")
        down = linear(gen, up.out, case["wt"], case["k"])
        calls, keep, out = [up.call, down.call], [up, down], [up.out, down.out]
    elif kind == "layer":
        wt, rows, heads, head_dim = case["wt"], case["rows"], case["heads"], case["head_dim"]
        width, keys = heads * head_dim, case["past"] + case["rows"]
        x = normal(gen, (rows, width), "f16")
        for _ in range(case["layers"]):
            qkv = linear(gen, x, wt, 3 * width)
            caches = [normal(gen, (1, heads, keys, head_dim), "f16") for _ in range(2)]
            row = (ctypes.c_int64 * 3)(rows * 3 * width, head_dim, 3 * width)
            base = qkv.out.data_ptr()
            write = (ra.lib().rt_cache_write_kv_enqueue, (device().ctx, _ffi.RT_F16, ptr(caches[0]), base + 2 * width, ptr(caches[1]), base + 4 * width, row,
                                                          1, heads, keys, case["past"], rows, head_dim))
            a = torch.empty((rows, width), dtype=torch.float16, device=GPU)
            desc = attention_desc(heads, head_dim, rows, keys, list(row), [heads * keys * head_dim, keys * head_dim, head_dim], True)
            attend, alive = attention_call(desc, base, caches[0], caches[1], None, a)
            o, up = linear(gen, a, wt, width), linear(gen, x, wt, 4 * width, "gelu")
            down = linear(gen, up.out, wt, width, scale=1.5)  # the layers' outputs keep the size of their inputs
            calls += [qkv.call, write, attend, o.call, up.call, down.call]
            keep += [qkv, row, caches, alive, o, up, down]
            out += [qkv.out, a, o.out, down.out]
            x = down.out
    elif kind == "nn":
        wt, rows, heads, head_dim = case["wt"], case["rows"], case["heads"], case["head_dim"]
        width, keys = heads * head_dim, case["past"] + case["rows"]

        def module(n, k, scale=1.0):
            return ra.nn.Linear(tensor(weight(gen, n, k, wt, scale), (n, k), wt), tensor(normal(gen, (n,), "f16") * 0.02, (n,), "f16"))

        q, k, v, o = (module(width, width) for _ in range(4))
        mlp = ra.nn.MLP(module(4 * width, width), module(width, 4 * width))
        cache = ra.nn.KVEntry(*(tensor(normal(gen, (1, heads, keys, head_dim), "f16"), (1, heads, keys, head_dim), "f16") for _ in range(2)),
                              entries=case["past"])
        return {"attn": ra.nn.SelfAttention(q, k, v, o, heads), "mlp": mlp, "cache": cache,
                "x": tensor(normal(gen, (1, rows, width), "f16"), (1, rows, width), "f16")}
    elif kind == "attention":
        heads, head_dim, rows, keys = case["heads"], case["head_dim"], case["rows"], case["keys"]
        q = normal(gen, (heads, rows, head_dim), "f16")
        k, v = (normal(gen, (heads, keys, head_dim), "f16") for _ in range(2))
        mask = None
        if case["mask"] in ("f32", "f16"):  # the reference's callers pass causality as a tensor of 0 and -inf
            hidden = torch.arange(keys, device=GPU)[None, :] > torch.arange(rows, device=GPU)[:, None] + (keys - rows)
            mask = torch.zeros((rows, keys), device=GPU).masked_fill_(hidden, float("-inf")).to(torch_type(case["mask"]))
        a = torch.empty((rows, heads * head_dim), dtype=torch.float16, device=GPU)
        desc = attention_desc(heads, head_dim, rows, keys, [q.numel(), rows * head_dim, head_dim], [k.numel(), keys * head_dim, head_dim],
                              case["mask"] == "causal", mask)
        attend, alive = attention_call(desc, q, k, v, mask, a)
        calls, keep, out = [attend], [alive], [a]
    else:
        dt, heads, head_dim, rows, keys = case["dt"], case["heads"], case["head_dim"], case["rows"], case["keys"]
        # the scale of the scores rides on q, as whisper's module has it
        q = normal(gen, (heads, rows, head_dim), dt) / math.sqrt(head_dim)
        v = normal(gen, (heads, keys, head_dim), dt)
        if dt == "f32":  # the f32 modules permute the keys beforehand
            scores = Product(q, dt, q.shape, normal(gen, (heads, head_dim, keys), dt), dt, (heads, head_dim, keys))
        else:
            scores = Product(q, dt, q.shape, normal(gen, (heads, keys, head_dim), dt), dt, (heads, keys, head_dim), trans_rhs=True)
        shape = (ctypes.c_int64 * 3)(heads, rows, keys)
        softmax = (ra.lib().rt_softmax_enqueue, (device().ctx, int(DT[dt]), ptr(scores.out), 3, shape, 2))
        values = Product(scores.out, dt, scores.out.shape, v, dt, v.shape)
        calls, keep, out = [scores.call, softmax, values.call], [scores, shape, values], [scores.out, values.out]
    return {"calls": calls, "keep": keep, "out": out}


def run(state):
    if "attn" in state:
        a = state["attn"].schedule(state["x"], state["cache"])
        y = state["mlp"].schedule(a).resolve()
        return [t.storage.view(torch.float16)[: t.numel()].view(t.shape) for t in (a, y)]
    stream = torch.cuda.current_stream().cuda_stream
    for enqueue, args in state["calls"]:
        check(enqueue(*args, stream))
    return state["out"]


# ---- what a pass cannot do without, and how exact its results are ------------------------------------------------------


def work(case):
    kind = case["kind"]

    def product(rows, n, k, wt):
        e = 4 if activation_type(wt) == "f32" else 2
        return n * k * BITS[wt] / 8 + (rows * k + n + rows * n) * e, 2.0 * rows * n * k

    def attention(heads, head_dim, rows, keys, causal, mask_bytes=0):
        seen = keys - (rows - 1) / 2 if causal else keys  # keys a query sees, on average
        return 2 * heads * head_dim * 2 * (rows + keys) + rows * keys * mask_bytes, 4.0 * heads * head_dim * rows * seen

    if kind == "linear":
        parts = [product(case["rows"], case["n"], case["k"], case["wt"])]
    elif kind == "mlp":
        parts = [product(case["rows"], case["n"], case["k"], case["wt"]), product(case["rows"], case["k"], case["n"], case["wt"])]
    elif kind in ("layer", "nn"):
        rows, width, wt = case["rows"], case["heads"] * case["head_dim"], case["wt"]
        parts = [product(rows, 3 * width, width, wt), product(rows, width, width, wt), product(rows, 4 * width, width, wt), product(rows, width, 4 * width, wt),
                 attention(case["heads"], case["head_dim"], rows, case["past"] + rows, True), (8.0 * rows * width, 0)]
        parts = parts * case.get("layers", 1)
    elif kind == "attention":
        parts = [attention(case["heads"], case["head_dim"], case["rows"], case["keys"], case["mask"] in ("causal", "f32", "f16"),
                           {"f32": 4, "f16": 2}.get(case["mask"], 0))]
    else:
        h, d, r, k, e = case["heads"], case["head_dim"], case["rows"], case["keys"], 4 if case["dt"] == "f32" else 2
        # the scores are written, read and written by the softmax and read once more: three operators
        parts = [(e * h * (r * d + k * d + r * k), 2.0 * h * r * k * d), (2.0 * e * h * r * k, 0), (e * h * (r * k + k * d + r * d), 2.0 * h * r * k * d)]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    # Measured against float64 over the listed cases and two dozen drawn ones: f32 up to 1.3e-6 (largest single value 7e-6), growing
    # with the square root of K, which reaches four times what was drawn there; f16 up to 6.4e-4 (1e-2), the roundings of a layer's
    # intermediate results.  About four times that.
    f32 = case.get("wt") in ("f32", "q8_0f") or case.get("dt") == "f32"
    return {"rel": 8e-6, "max": 5e-5} if f32 else {"rel": 2.5e-3, "max": 4e-2}
