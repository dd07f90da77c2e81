"""The calls whose time this repository looks after: matrix products as programs
make them through gemmkit_amd's entry points, from single-row decode steps to
full 4096^3 products, in float32, bfloat16 and int8.

Layouts are three letters for A, B and C, each "r" (row-major) or "c"
(column-major): "rrr" is the plain row-major call, "rcr" a weight stored
output-major and read transposed (x @ W^T), "ccc" the column-major libraries'
call.  Calls are stream-ordered (set_synchronous(False)), as a program that
issues many of them would have it.
"""
import math

import torch

import gemmkit_amd as gk

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "i8": torch.int8}
ESIZE = {"f32": 4, "bf16": 2, "i8": 1}


def _gemm(name, dtype, m, k, n, layout, **more):
    return dict(name=name, op="gemm", dtype=dtype, m=m, k=k, n=n, batch=1, layout=layout, **more)


def listed():
    return [
        # The library's own quick-start size: a small dense row-major product,
        # where launches and memory latency are the whole time.
        _gemm("f32_512", "f32", 512, 512, 512, "rrr"),
        # An ordinary single-precision product, everything row-major.
        _gemm("f32_2048", "f32", 2048, 2048, 2048, "rrr"),
        # Many small products of one shape whose sides are no tile's multiple
        # (per-sample transforms, blocks of a block-diagonal system).
        dict(name="f32_batched", op="batched", dtype="f32", m=200, k=150, n=120, batch=96,
             layout="rrr"),
        # The largest plain int8 product: weight read transposed, int32 sums out.
        _gemm("i8_4096", "i8", 4096, 4096, 4096, "rcr"),
        # A quantized linear layer at prefill: prepacked weight, per-channel
        # scale and bias, ReLU, int8 out.
        dict(name="i8_layer", op="layer", dtype="i8", m=2048, k=4096, n=11008, batch=1,
             layout="rcr"),
        # A bfloat16 linear layer at prefill with its bias and ReLU fused, the
        # weight stored input-major as most training code holds it.
        dict(name="bf16_fused", op="fused", dtype="bf16", m=2048, k=4096, n=4096, batch=1,
             layout="rrr"),
        # Attention scores: 64 heads' Q K^T, float32 out.
        dict(name="bf16_attn", op="scores", dtype="bf16", m=512, k=128, n=512, batch=64,
             layout="rcr"),
        # A bfloat16 product with no aligned side, as data-dependent sizes give.
        _gemm("bf16_ragged", "bf16", 777, 1001, 1501, "rrr"),
        # One decode step through a quantized projection (one token).
        _gemm("i8_decode", "i8", 1, 4096, 14336, "rcr"),
        # The same for a batch of eight sequences.
        _gemm("i8_decode8", "i8", 8, 4096, 14336, "rcr"),
        # A large dense matrix times a vector (iterative solvers).
        _gemm("f32_matvec", "f32", 16384, 16384, 1, "rrr"),
        # One decode step in bfloat16 with the weight stored input-major.
        _gemm("bf16_decode_row", "bf16", 1, 4096, 11008, "rrr"),
    ]


def _side(rng, lo, hi):
    """A size in [lo, hi], spread over its logarithm; two thirds are multiples
    of 8 or 64, the rest whatever comes, odd ones among them."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice((1, 8, 64))
    return max(lo, min(hi, (v + step // 2) // step * step if v >= step else v))


def draw(rng):
    op = rng.choice(("gemm", "gemm", "batched", "vector", "vector", "layer", "fused", "scores",
                     "packed"))
    layout = rng.choice(("rrr", "rcr", "ccc"))
    if op in ("gemm", "fused"):
        dtype = rng.choice(("f32", "bf16", "i8") if op == "gemm" else ("f32", "bf16"))
        most = 2 * 2048 ** 3 if dtype == "f32" else 2 * 4096 ** 3
        while True:
            m, k, n = (_side(rng, 64, 4096) for _ in range(3))
            if 2 * m * k * n <= most:
                return dict(op=op, dtype=dtype, m=m, k=k, n=n, batch=1, layout=layout)
    if op == "batched":
        dtype = rng.choice(("f32", "bf16"))
        while True:
            m, k, n = (_side(rng, 16, 512) for _ in range(3))
            batch = _side(rng, 4, 256)
            if 2 * m * k * n * batch <= 2 ** 33:
                return dict(op=op, dtype=dtype, m=m, k=k, n=n, batch=batch, layout=layout)
    if op == "vector":  # decode steps and matrix-vector products
        dtype = rng.choice(("f32", "bf16", "i8"))
        few, k, n = rng.choice((1, 1, 2, 4, 8, 16)), _side(rng, 1024, 16384), _side(rng, 1024, 16384)
        if layout == "rrr" and rng.random() < 0.3:
            return dict(op="gemm", dtype=dtype, m=n, k=k, n=few, batch=1, layout=layout)
        return dict(op="gemm", dtype=dtype, m=few, k=k, n=n, batch=1, layout=layout)
    if op == "layer":
        return dict(op=op, dtype="i8", m=_side(rng, 16, 2048), k=_side(rng, 512, 4096),
                    n=_side(rng, 512, 11008), batch=1, layout="rcr")
    if op == "scores":
        return dict(op=op, dtype="bf16", m=_side(rng, 64, 512), k=rng.choice((64, 96, 128)),
                    n=_side(rng, 64, 512), batch=_side(rng, 8, 64), layout="rcr")
    # a few rows against a prepacked weight, column-major C
    return dict(op="packed", dtype=rng.choice(("f32", "bf16", "i8")), m=_side(rng, 8, 256),
                k=_side(rng, 512, 4096), n=_side(rng, 512, 4096), batch=1,
                layout=rng.choice(("rrc", "rcc", "ccc")))


def _strides(letter, rows, cols):
    return (cols, 1) if letter == "r" else (1, rows)


def _values(case, seed):
    """A and B (flat, in the layout's order), and the bias and scales where the
    call has them."""
    m, k, n, batch, dtype = case["m"], case["k"], case["n"], case["batch"], case["dtype"]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(count, std=1.0):
        return torch.randn(count, generator=g, device="cuda").mul_(std).to(DTYPES[dtype])

    def ints(count, lo, hi, dt):
        return torch.randint(lo, hi + 1, (count,), generator=g, device="cuda", dtype=dt)

    v = {}
    if dtype == "i8":
        lo = -127 if case["op"] == "layer" else -128
        v["a"], v["b"] = ints(batch * m * k, lo, 127, torch.int8), ints(batch * k * n, lo, 127, torch.int8)
    elif case["op"] == "scores":
        v["a"], v["b"] = normal(batch * m * k), normal(batch * k * n)
    else:  # activations against weights of the usual initial scale
        v["a"], v["b"] = normal(batch * m * k), normal(batch * k * n, 1.0 / math.sqrt(k))
    if case["op"] == "fused":
        v["bias"] = normal(n)
    if case["op"] == "layer":
        v["bias"] = ints(n, -65536, 65536, torch.int32)
        v["scales"] = torch.empty(n, device="cuda").uniform_(1e-4, 1e-2, generator=g)
    return v


def _out_dtype(case):
    if case["op"] == "layer":
        return torch.int8
    if case["dtype"] == "i8":
        return torch.int32
    return torch.float32 if case["op"] == "scores" else DTYPES[case["dtype"]]


def prepare(case, seed):
    gk.set_synchronous(False)
    m, k, n, batch = case["m"], case["k"], case["n"], case["batch"]
    la, lb, lc = case["layout"]
    v = _values(case, seed)
    out = torch.zeros(batch * m * n, dtype=_out_dtype(case), device="cuda")
    s = dict(case=case, out=out, values=v,
             a=gk.MatRef(v["a"], m, k, *_strides(la, m, k)),
             b=gk.MatRef(v["b"], k, n, *_strides(lb, k, n)),
             c=gk.MatMut(out, m, n, *_strides(lc, m, n)))
    if case["op"] == "layer":
        s["packed"] = gk.prepack_rhs_i8(s["b"])
        s["req"] = gk.Requantize(gk.RequantScale.PerCol(v["scales"]), 0, v["bias"],
                                 bias_axis="col", relu=True)
    elif case["op"] == "packed":
        s["packed"] = (gk.prepack_rhs_i8 if case["dtype"] == "i8" else gk.prepack_rhs)(s["b"])
    elif case["op"] == "fused":
        s["bias"] = gk.Bias.PerCol(v["bias"])
    return s


def run(s):
    case = s["case"]
    op, m, k, n = case["op"], case["m"], case["k"], case["n"]
    if op == "gemm":
        if case["dtype"] == "i8":
            gk.gemm_i8(1, s["a"], s["b"], 0, s["c"])
        else:
            gk.gemm(1.0, s["a"], s["b"], 0.0, s["c"])
    elif op == "fused":
        gk.gemm_fused(1.0, s["a"], s["b"], 0.0, s["c"], bias=s["bias"], act=gk.Activation.Relu)
    elif op == "batched":
        gk.gemm_batched(case["batch"], 1.0, s["a"], m * k, s["b"], k * n, 0.0, s["c"], m * n)
    elif op == "scores":
        gk.gemm_batched_bf16_f32out(case["batch"], 1.0 / math.sqrt(k), s["a"], m * k, s["b"],
                                    k * n, 0.0, s["c"], m * n)
    elif op == "layer":
        # scales were checked when the layer was loaded: the serving loop takes the raw entry
        v = s["values"]
        gk.gemm_i8_packed_b_requant_unchecked(m, v["a"], k, 1, s["packed"], 0.0, v["scales"], 0,
                                              v["bias"], s["out"], n, 1, axis=1, relu=True)
    elif case["dtype"] == "i8":
        gk.gemm_i8_packed_b(1, s["a"], s["packed"], 0, s["c"])
    else:
        gk.gemm_packed_b(1.0, s["a"], s["packed"], 0.0, s["c"])
    return s["out"]


def work(case):
    m, k, n, batch, e = case["m"], case["k"], case["n"], case["batch"], ESIZE[case["dtype"]]
    size = torch.empty((), dtype=_out_dtype(case)).element_size()
    extra = {"fused": n * e, "layer": 8 * n}.get(case["op"], 0)
    return {"bytes": batch * ((m * k + k * n) * e + m * n * size) + extra,
            "flops": 2 * batch * m * k * n}


def tolerance(case):
    if case["dtype"] == "i8":
        return "exact"
    if _out_dtype(case) == torch.bfloat16:
        return {"rel": 7e-3}  # one bfloat16 rounding of a float32 sum: 1.7e-3 seen
    return {"rel": 4e-6}  # float32 sums of up to 16384 terms: up to 1e-6 seen


def exact(case, seed):
    m, k, n, batch = case["m"], case["k"], case["n"], case["batch"]
    la, lb, lc = case["layout"]
    v = _values(case, seed)

    def full(flat, letter, rows, cols):
        t = flat.view(batch, rows, cols) if letter == "r" else flat.view(batch, cols, rows).mT
        return t.double().contiguous()

    c = torch.matmul(full(v["a"], la, m, k), full(v["b"], lb, k, n))
    if case["op"] == "scores":
        c *= 1.0 / math.sqrt(k)
    if case["op"] == "fused":
        c = (c + v["bias"].double()).clamp_(min=0.0)
    if case["op"] == "layer":
        c = torch.round((c + v["bias"].double()) * v["scales"].double()).clamp_(0, 127)
    if lc == "c":
        c = c.mT.contiguous()
    c = c.reshape(-1)
    return c.to(_out_dtype(case)) if case["dtype"] == "i8" else c
