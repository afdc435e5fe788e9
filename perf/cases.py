"""The work a program built on this library has it do, as measurable cases.

A case is a dict of plain values.  `listed()` names twelve of them, `draw(rng)` makes further ones of the same ranges;
`prepare` builds what a user's program holds before the call (inputs in device memory, weights, an execution plan),
`run` makes one pass through the public entry points, `work` states what the pass cannot do without and `tolerance` how
far two correct implementations at the same precision lie apart.

Two ways of calling are covered, because both are in use: a plan made once with `Tensor.prepare()` and executed per pass
(an inference loop over fixed shapes), and a lazy graph built anew and realized on every pass (a script, a decode step whose
shapes grow by one token).
"""
import math

import numpy as np
import torch

from morok_amd import uop
from morok_amd.decoder import DecoderBlock
from morok_amd.device import Buffer
from morok_amd.tensor import Tensor

# name in a case -> (tag of the library, torch dtype, bytes, type string of the array interface)
_TYPES = {"f32": (uop.F32, torch.float32, 4, "<f4"), "f16": (uop.F16, torch.float16, 2, "<f2"), "bf16": (uop.BF16, torch.bfloat16, 2, "<i2"),
          "i32": (uop.I32, torch.int32, 4, "<i4"), "bool": (uop.BOOL, torch.uint8, 1, "|u1")}


class _Memory:
    """A library buffer as torch sees it; the torch tensor keeps this object, and so the buffer, alive."""

    def __init__(self, buf, shape, dtype):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": _TYPES[dtype][3], "data": (buf.ptr, False), "version": 2, "strides": None}


def _view(buf, shape, dtype):
    """The buffer's memory as a torch tensor (no copy)."""
    t = torch.as_tensor(_Memory(buf, shape, dtype), device="cuda")
    return t.view(torch.bfloat16) if dtype == "bf16" else t


def _device(shape, dtype):
    """A library tensor over fresh device memory, and the same memory as a torch tensor to fill."""
    buf = Buffer(int(math.prod(shape)) * _TYPES[dtype][2]).ensure_allocated()
    return Tensor.from_buffer(buf, shape, _TYPES[dtype][0]), _view(buf, shape, dtype)


class _Inputs:
    """Seeded inputs in device memory."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, shape, dtype, sigma=1.0, mean=0.0):
        t, mem = _device(shape, dtype)
        mem.normal_(mean, sigma, generator=self.gen)
        return t

    def uniform(self, shape, dtype, lo=-1.0, hi=1.0):
        t, mem = _device(shape, dtype)
        mem.uniform_(lo, hi, generator=self.gen)
        return t

    def randint(self, shape, high):
        t, mem = _device(shape, "i32")
        mem.random_(0, high, generator=self.gen)
        return t

    def padding_mask(self, rows, keys):
        """A Bool key-padding mask [rows, 1, 1, keys] of sequences of different lengths (half of the keys to all of them)."""
        t, mem = _device((rows, 1, 1, keys), "bool")
        length = torch.randint(max(1, keys // 2), keys + 1, (rows, 1, 1, 1), generator=self.gen, device="cuda")
        mem.copy_((torch.arange(keys, device="cuda") < length).to(torch.uint8))
        return t

    def host_bf16(self, shape, sigma, mean=0.0):
        """bf16 bit patterns in host memory, as a checkpoint loader hands them over."""
        x = torch.empty(shape, dtype=torch.bfloat16, device="cuda").normal_(mean, sigma, generator=self.gen)
        return x.view(torch.int16).cpu().numpy().view(np.uint16)


# ---------------------------------------------------------------------------------------------- the cases
def listed():
    return [
        # smallest: a two-layer f32 classifier over a small batch, written with tensor ops and realized each time
        {"name": "classifier_64", "kind": "classifier", "batch": 64, "features": 784, "hidden": 256, "classes": 10},
        # the f32 product of the benchmark (plan executed per pass)
        {"name": "matmul_f32_1024", "kind": "matmul_f32", "m": 1024, "n": 1024, "k": 1024},
        # the row softmax of the benchmark: one pass over 512 MiB
        {"name": "softmax_8192", "kind": "softmax", "rows": 8192, "cols": 8192, "dtype": "f32"},
        # RMSNorm with gain over the tokens of a prefill
        {"name": "rmsnorm_8192x4096", "kind": "rmsnorm", "rows": 8192, "cols": 4096},
        # the bf16 product of the benchmark, [K, N] weight
        {"name": "gemm_bf16_4096", "kind": "product", "m": 4096, "n": 4096, "k": 4096, "dtype": "bf16", "layout": "kn", "bias": False},
        # vocabulary projection over an odd vocabulary, weight as a Linear layer stores it
        {"name": "vocab_head_50257", "kind": "product", "m": 512, "n": 50257, "k": 768, "dtype": "bf16", "layout": "nt", "bias": False},
        # a Linear layer with bias in half precision over a ragged number of rows
        {"name": "linear_f16_1000", "kind": "product", "m": 1000, "n": 3000, "k": 2048, "dtype": "f16", "layout": "nt", "bias": True},
        # causal attention of the benchmark, the largest single kernel
        {"name": "attention_causal_4096", "kind": "attention", "batch": 8, "kv_heads": 32, "group": 1, "sq": 4096, "sk": 4096, "d": 128, "causal": True,
         "mask": False},
        # an encoder's attention over a batch of sequences of different lengths (key-padding mask), head dim 64
        {"name": "attention_padded_1000", "kind": "attention", "batch": 8, "kv_heads": 16, "group": 1, "sq": 1000, "sk": 1000, "d": 64, "causal": False,
         "mask": True},
        # one new query per head against a cache of 4096 keys
        {"name": "attention_decode_4096", "kind": "attention", "batch": 1, "kv_heads": 32, "group": 1, "sq": 1, "sk": 4096, "d": 128, "causal": False,
         "mask": False},
        # the decoder block of the benchmark, prefill of 4 x 2048 tokens
        {"name": "decoder_prefill_4x2048", "kind": "prefill", "batch": 4, "seq": 2048, "hidden": 4096, "ffn": 11008},
        # one decode step of 8 sequences through the same block over cached keys and values, built and realized anew as the cache grows
        {"name": "decoder_step_8x2047", "kind": "step", "batch": 8, "pos": 2047, "hidden": 4096, "ffn": 11008},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _aligned(rng, lo, hi, units=(64, 64, 8, 1)):
    """A size as layers have them: most are multiples of 64, some of 8, some are odd."""
    unit = rng.choice(units)
    return max(unit, _log(rng, lo, hi) // unit * unit)


_WIDTHS = ((1024, 2816), (2048, 5504), (4096, 11008))


def draw(rng):
    kind = rng.choice(("classifier", "matmul_f32", "softmax", "rmsnorm", "product", "product", "attention", "attention", "decode", "prefill", "step"))
    while True:
        if kind == "classifier":
            return {"kind": kind, "batch": _log(rng, 1, 512), "features": _log(rng, 16, 2048), "hidden": _log(rng, 32, 1024), "classes": _log(rng, 2, 1000)}
        if kind == "matmul_f32":
            return {"kind": kind, "m": _aligned(rng, 64, 1536, (64, 1)), "n": _aligned(rng, 64, 1536, (64, 1)), "k": _aligned(rng, 64, 1536, (64, 1))}
        if kind == "softmax":
            c = {"kind": kind, "rows": _log(rng, 16, 16384), "cols": _log(rng, 64, 65536), "dtype": rng.choice(("f32", "f32", "bf16"))}
            if c["rows"] * c["cols"] <= 1 << 26:
                return c
        elif kind == "rmsnorm":
            return {"kind": kind, "rows": _log(rng, 1, 16384), "cols": _aligned(rng, 256, 8192)}
        elif kind == "product":
            layout = rng.choice(("kn", "nt"))
            c = {"kind": kind, "m": _log(rng, 1, 8192), "n": _aligned(rng, 256, 52000), "k": _aligned(rng, 256, 12288, (64, 64, 64, 8, 1)),
                 "dtype": rng.choice(("bf16", "bf16", "f16")), "layout": layout, "bias": layout == "nt" and rng.random() < 0.5}
            if c["n"] * c["k"] <= 1 << 28 and c["m"] * c["n"] * c["k"] <= 1 << 39:
                return c
        elif kind == "attention":
            sq = _log(rng, 128, 8192)
            causal, mask = rng.choice(((True, False), (True, False), (False, False), (False, True)))
            sk = sq if causal else _log(rng, 128, 8192)
            if mask:
                sk = (sk + 7) // 8 * 8  # sequences are padded to a common multiple of eight
            c = {"kind": kind, "batch": _log(rng, 1, 16), "kv_heads": rng.choice((8, 16, 32)), "group": 1, "sq": sq, "sk": sk, "d": rng.choice((64, 128, 128, 256)),
                 "causal": causal, "mask": mask}
            if work(c)["flops"] <= 1.1e12:
                return c
        elif kind == "decode":
            mask = rng.random() < 0.3
            sk = _log(rng, 256, 32768)
            c = {"kind": "attention", "batch": _log(rng, 1, 32), "kv_heads": rng.choice((4, 8, 16, 32)), "group": rng.choice((1, 1, 4, 8)), "sq": 1,
                 "sk": (sk + 7) // 8 * 8 if mask else sk, "d": rng.choice((64, 128, 128, 256)), "causal": False, "mask": mask}
            if work(c)["bytes"] <= 2e9:
                return c
        elif kind == "prefill":
            hidden, ffn = rng.choice(_WIDTHS)
            c = {"kind": kind, "batch": _log(rng, 1, 8), "seq": _log(rng, 64, 2048), "hidden": hidden, "ffn": ffn}
            if c["batch"] * c["seq"] <= 8192:
                return c
        else:
            hidden, ffn = rng.choice(_WIDTHS)
            c = {"kind": "step", "batch": _log(rng, 1, 16), "pos": _log(rng, 127, 4095), "hidden": hidden, "ffn": ffn}
            if work(c)["bytes"] <= 2e9:
                return c


# ---------------------------------------------------------------------------------------------- one pass
def _attention_operands(case, inputs):
    """q, k, v and mask.  Grouped queries: the key heads ride on the batch axis and one key head is expanded over its group."""
    rows = case["batch"] * (case["kv_heads"] if case["group"] > 1 else 1)
    heads = case["group"] if case["group"] > 1 else case["kv_heads"]
    kv = 1 if case["group"] > 1 else heads
    q = inputs.normal((rows, heads, case["sq"], case["d"]), "bf16")
    k = inputs.normal((rows, kv, case["sk"], case["d"]), "bf16")
    v = inputs.normal((rows, kv, case["sk"], case["d"]), "bf16")
    if case["group"] > 1:
        full = [rows, heads, case["sk"], case["d"]]
        k, v = k.try_expand(full), v.try_expand(full)
    return q, k, v, inputs.padding_mask(rows, case["sk"]) if case["mask"] else None


def _block_weights(case, inputs, linear_layout):
    """Random-init weights of one decoder block, scaled so that activations stay of order one.  Projections are made in the
    layout the block keeps ([in, out], or a Linear layer's [out, in]), so that it takes them without transposing."""
    h, f, vocab = case["hidden"], case["ffn"], 32000
    shapes = {"Wq": (h, h), "Wk": (h, h), "Wv": (h, h), "Wo": (h, h), "W1": (h, f), "W3": (h, f), "W2": (f, h)}
    w = {"emb": inputs.host_bf16((vocab, h), 1.0), "w_an": inputs.host_bf16((h,), 0.1, 1.0), "w_fn": inputs.host_bf16((h,), 0.1, 1.0)}
    for name, (i, o) in shapes.items():
        w[name] = inputs.host_bf16((o, i), i ** -0.5).T if linear_layout else inputs.host_bf16((i, o), i ** -0.5)
    return w


def _planned(root, shape, dtype, keep):
    """A program that prepares its graph once and executes the plan per pass."""
    plan = root.prepare()
    return {"plan": plan, "out": _view(root.buffer(), shape, dtype), "keep": keep}


def prepare(case, seed):
    inputs, kind = _Inputs(seed), case["kind"]
    if kind == "classifier":
        b, f, h, c = case["batch"], case["features"], case["hidden"], case["classes"]
        s = {"x": inputs.normal((b, f), "f32"), "w1": inputs.normal((h, f), "f32", f ** -0.5), "b1": inputs.normal((h,), "f32", 0.1),
             "w2": inputs.normal((c, h), "f32", h ** -0.5), "b2": inputs.normal((c,), "f32", 0.1)}
    elif kind == "matmul_f32":
        m, n, k = case["m"], case["n"], case["k"]
        a, b = inputs.uniform((m, k), "f32"), inputs.uniform((k, n), "f32")
        s = _planned(a.matmul(b), (m, n), "f32", (a, b))
    elif kind == "softmax":
        x = inputs.normal((case["rows"], case["cols"]), case["dtype"], 2.0)
        s = _planned(x.softmax(-1), x.shape, case["dtype"], x)
    elif kind == "rmsnorm":
        x, g = inputs.normal((case["rows"], case["cols"]), "bf16"), inputs.normal((case["cols"],), "bf16", 0.1, 1.0)
        s = _planned(x.rms_norm(-1, 1e-6).try_mul(g).cast(uop.BF16), x.shape, "bf16", (x, g))
    elif kind == "product":
        m, n, k, dt = case["m"], case["n"], case["k"], case["dtype"]
        x = inputs.normal((m, k), dt)
        w = inputs.normal((n, k) if case["layout"] == "nt" else (k, n), dt, k ** -0.5)
        b = inputs.normal((n,), dt) if case["bias"] else None
        s = _planned(x.linear(w, b) if case["layout"] == "nt" else x.matmul(w), (m, n), dt, (x, w, b))
    elif kind == "attention":
        q, k, v, mask = _attention_operands(case, inputs)
        s = _planned(q.scaled_dot_product_attention(k, v, is_causal=case["causal"], attn_mask=mask), q.shape, "bf16", (q, k, v, mask))
    elif kind == "prefill":
        tokens, hidden = case["batch"] * case["seq"], case["hidden"]
        block = DecoderBlock(_block_weights(case, inputs, False), case["batch"], case["seq"], hidden, hidden // 128, case["ffn"], eps=1e-6)
        ids = inputs.randint((tokens,), 32000)
        torch.cuda.synchronize()
        s = _planned(block.forward(ids), (tokens, hidden), "bf16", (block, ids))
    else:
        b, hidden = case["batch"], case["hidden"]
        block = DecoderBlock(_block_weights(case, inputs, True), b, 1, hidden, hidden // 128, case["ffn"], eps=1e-6, linear_layout=True)
        past = (b, hidden // 128, case["pos"], 128)
        s = {"block": block, "ids": inputs.randint((b,), 32000), "k": inputs.normal(past, "bf16"), "v": inputs.normal(past, "bf16"), "pos": case["pos"]}
    torch.cuda.synchronize()  # the inputs are written on torch's stream, the library runs on its own
    return s


def run(state):
    if "plan" in state:
        state["plan"].execute()
        return state["out"]
    if "block" in state:
        out, k, v = state["block"].decode_step(state["ids"], state["k"], state["v"], state["pos"])
        return [_view(t.realize().buffer(), t.shape, "bf16") for t in (out, k, v)]
    hidden = state["x"].linear(state["w1"], state["b1"]).maximum(0.0)
    y = hidden.linear(state["w2"], state["b2"]).log_softmax(-1).realize()
    return _view(y.buffer(), y.shape, "f32")


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "classifier":
        b, f, h, c = case["batch"], case["features"], case["hidden"], case["classes"]
        return {"bytes": 4.0 * (b * f + h * f + h + c * h + c + b * c), "flops": 2.0 * b * h * (f + c)}
    if kind == "matmul_f32":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4.0 * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 2.0 * n * _TYPES[case["dtype"]][2], "flops": 4.0 * n}
    if kind == "rmsnorm":
        n = case["rows"] * case["cols"]
        return {"bytes": 4.0 * n + 2.0 * case["cols"], "flops": 4.0 * n}
    if kind == "product":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2.0 * (m * k + k * n + m * n + (n if case["bias"] else 0)), "flops": 2.0 * m * n * k}
    if kind == "attention":
        pairs = case["batch"] * case["kv_heads"]
        scores = pairs * case["group"] * case["sq"] * case["sk"] * (0.5 if case["causal"] else 1.0)
        read = 2.0 * pairs * (2 * case["group"] * case["sq"] + 2 * case["sk"]) * case["d"]
        rows = case["batch"] * (case["kv_heads"] if case["group"] > 1 else 1)
        return {"bytes": read + (rows * case["sk"] if case["mask"] else 0), "flops": 4.0 * scores * case["d"]}
    h, f = case["hidden"], case["ffn"]
    weights = 2.0 * (4 * h * h + 3 * h * f + 2 * h)
    if kind == "prefill":
        t = case["batch"] * case["seq"]
        return {"bytes": weights + 2.0 * 2 * t * h + 4.0 * t, "flops": 2.0 * t * h * (4 * h + 3 * f) + 2.0 * t * case["seq"] * h}
    b, pos = case["batch"], case["pos"]
    # the weights, the past read once, the grown keys and values written once
    return {"bytes": weights + 2.0 * 2 * b * h * (2 * pos + 1) + 2.0 * 2 * b * h, "flops": 2.0 * b * h * (4 * h + 3 * f) + 4.0 * b * h * (pos + 1)}


def tolerance(case):
    """About four times what each path measured against itself in 64 bits (2-norm): one rounding to bf16 1.7e-3, to f16 2.7e-4; attention, which
    rounds its weights to bf16 as well, 2.0e-3 to 2.3e-3; a whole block 3.6e-3; f32 sums over 1024 products in order 5.7e-7; f32 softmax 1e-7."""
    kind = case["kind"]
    if kind in ("classifier", "matmul_f32"):
        return {"rel": 3e-6}
    if kind == "attention":
        return {"rel": 9e-3}
    if kind in ("prefill", "step"):
        return {"rel": 1.4e-2}
    return {"rel": {"f32": 1e-6, "f16": 1.2e-3, "bf16": 6.5e-3}[case.get("dtype", "bf16")]}
