"""The work whose speed is tracked: what a program that uses this package has it do.

A case is a dict of plain values; `kind` picks one of the paths below, the
rest gives its sizes, code format and input type.

  roundtrip  a tensor packed and unpacked again: mx_tensor.quantize, dequantize
  kv         one decode step of a windowed KV cache: append_kv, then get
  matmul     the packed product qa @ qb, from packed operands or from floats (mx_matmul)
  linear     one mx_linear
  mlp        two mx_linear with a SiLU between them (a Sequential after to_mx)
  dynamic    an mx_dynamic_linear and the gradient of its input
  int8       per-token activation codes, then the int8 x int8 linear

A linear or mlp with `graph` runs as a captured graph's replay, the way a
decode loop runs it; the others are eager calls.
"""
import math

import torch
import torch.nn as nn
import torch.nn.functional as F

import qtpytorch_amd as qa

DEV = "cuda"
SRC = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
SEED_H = 1534857261  # rotation seed of the 'h' formats


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest product that is worth packing: two float operands of a
        # few hundred rows, packed and multiplied; launches and host work
        {"name": "matmul-512", "kind": "matmul", "m": 512, "k": 512, "n": 512, "dtype": "int8d", "block": 128,
         "floats": True},
        # packed 4-bit operands of a size between the small and the large
        # kernels, with ragged rows and columns
        {"name": "matmul-ragged", "kind": "matmul", "m": 1500, "k": 2048, "n": 1800, "dtype": "int4d", "block": 128,
         "floats": False},
        # the block the published int8 products were timed with, on a square
        # of ordinary size
        {"name": "matmul-block64", "kind": "matmul", "m": 2048, "k": 2048, "n": 2048, "dtype": "int8d", "block": 64,
         "floats": False},
        # the large packed product
        {"name": "matmul-8192", "kind": "matmul", "m": 8192, "k": 8192, "n": 8192, "dtype": "int8d", "block": 128,
         "floats": False},
        # a large weight (an odd number of rows) packed for storage and read back
        {"name": "roundtrip-int4", "kind": "roundtrip", "rows": 16383, "cols": 4096, "dtype": "int4d", "src": "fp32",
         "block": 128},
        # a square weight packed with the rotation of its rows
        {"name": "roundtrip-rotated", "kind": "roundtrip", "rows": 4096, "cols": 4096, "dtype": "int4dh",
         "src": "bf16", "block": 128},
        # a decode step over a full window of 2048 steps, 8 sequences of 32 heads
        {"name": "kv-window", "kind": "kv", "batch": 8, "heads": 32, "dim": 128, "steps": 2048, "dtype": "int8dv",
         "src": "fp16"},
        # a decoder's feed-forward pair for a small decode batch, replayed
        {"name": "mlp-decode", "kind": "mlp", "tokens": 8, "d": 4096, "f": 14336, "dtype": "int4d", "src": "bf16",
         "graph": True},
        # the same at a batch between decode and prefill (several sequences,
        # or drafted tokens that are verified together), 8-bit weights
        {"name": "mlp-batch", "kind": "mlp", "tokens": 48, "d": 8192, "f": 8192, "dtype": "int8d", "src": "fp32",
         "graph": True},
        # an output head whose width is no multiple of a block, decode batch
        {"name": "head-odd", "kind": "linear", "tokens": 16, "k": 4096, "n": 50257, "dtype": "int8d", "src": "bf16",
         "graph": False},
        # adapter training through a packed layer: prefill-sized forward and input gradient
        {"name": "dynamic-train", "kind": "dynamic", "tokens": 2048, "k": 4096, "n": 4096, "dtype": "int4d",
         "src": "bf16"},
        # prefill with 8-bit activations and weights
        {"name": "int8-prefill", "kind": "int8", "tokens": 4000, "k": 4096, "n": 4096, "src": "bf16"},
    ]


def _log(rng, lo, hi, step=1):
    """A size from lo to hi, even over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(["roundtrip", "kv", "matmul", "matmul", "linear", "linear", "mlp", "dynamic", "int8"])
    src = rng.choice(["fp32", "fp16", "bf16"])
    if kind == "roundtrip":
        dtype = rng.choice(["int8d", "int4d", "int2d", "float4d", "float8d", "int8dv", "int4dh", "int8dh"])
        cols = rng.choice([128, 512, 1024, 2048, 4096, 8192]) if dtype.endswith("h") else _log(rng, 96, 8192)
        total = _log(rng, 1 << 18, 1 << 26)
        return {"kind": kind, "rows": max(1, total // cols), "cols": cols, "dtype": dtype, "src": src, "block": 128}
    if kind == "kv":
        return {"kind": kind, "batch": rng.choice([1, 2, 4, 8]), "heads": rng.choice([8, 16, 32]),
                "dim": rng.choice([64, 128]), "steps": _log(rng, 64, 2048), "dtype": rng.choice(["int8d", "int8dv", "int4d"]),
                "src": src}
    if kind == "matmul":
        step = rng.choice([1, 8, 128])
        return {"kind": kind, "m": _log(rng, 64, 4096, step), "k": _log(rng, 256, 4096, rng.choice([8, 128, 128])),
                "n": _log(rng, 64, 4096, rng.choice([1, 16, 128])), "dtype": rng.choice(["int8d", "int8d", "int4d"]),
                "block": rng.choice([128, 128, 64]), "floats": rng.random() < 0.4}
    if kind == "linear":
        tokens = _log(rng, 1, 2048)
        return {"kind": kind, "tokens": tokens, "k": _log(rng, 512, 8192, 64),
                "n": _log(rng, 512, 32768, rng.choice([1, 128])),
                "dtype": rng.choice(["int4d", "int4d", "int8d", "float4d", "float8d"]), "src": src,
                "graph": tokens <= 64}
    if kind == "mlp":
        tokens = _log(rng, 1, 2048)
        return {"kind": kind, "tokens": tokens, "d": _log(rng, 1024, 8192, 128), "f": _log(rng, 2048, 14336, 128),
                "dtype": rng.choice(["int4d", "int4d", "int8d", "float4d"]), "src": src, "graph": tokens <= 64}
    if kind == "dynamic":
        return {"kind": kind, "tokens": _log(rng, 8, 2048), "k": _log(rng, 512, 8192, 128),
                "n": _log(rng, 512, 8192, 128), "dtype": rng.choice(["int4d", "int8d"]), "src": src}
    return {"kind": "int8", "tokens": _log(rng, 8, 4096), "k": _log(rng, 512, 8192, 64), "n": _log(rng, 512, 8192, 8),
            "src": src}


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _activations(g, shape, src):
    """Normal activations with a few large ones, as they meet a packed layer."""
    x = torch.randn(shape, generator=g, device=DEV)
    x[torch.rand(shape, generator=g, device=DEV) < 1e-3] *= 20.0
    return x.to(SRC[src])


def _weight(g, n, k):
    w = 0.02 * torch.randn(n, k, generator=g, device=DEV)
    w[torch.rand(n, k, generator=g, device=DEV) < 1e-3] *= 10.0
    return w


def _float_linear(weight, bias=None):
    lin = nn.Linear(weight.shape[1], weight.shape[0], bias=bias is not None, device="meta")
    lin.weight = nn.Parameter(weight, requires_grad=False)
    if bias is not None:
        lin.bias = nn.Parameter(bias, requires_grad=False)
    return lin


def _inputs(case, seed):
    """The float tensors of a case, in the order its state and its exact values take them."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "roundtrip":
        return [_activations(g, (case["rows"], case["cols"]), case["src"])]
    if kind == "kv":
        shape = (case["steps"] + 1, 2, case["batch"], case["heads"], 1, case["dim"])
        return [torch.randn(shape, generator=g, device=DEV, dtype=SRC[case["src"]])]
    if kind == "matmul":
        return [torch.randn(case["m"], case["k"], generator=g, device=DEV),
                torch.randn(case["k"], case["n"], generator=g, device=DEV)]
    if kind == "linear":
        return [_activations(g, (case["tokens"], case["k"]), case["src"]), _weight(g, case["n"], case["k"])]
    if kind == "mlp":
        return [_activations(g, (case["tokens"], case["d"]), case["src"]), _weight(g, case["f"], case["d"]),
                _weight(g, case["d"], case["f"])]
    x = _activations(g, (case["tokens"], case["k"]), case["src"])
    w = _weight(g, case["n"], case["k"])
    bias = 0.1 * torch.randn(case["n"], generator=g, device=DEV)
    if kind == "dynamic":
        return [x, w, bias, torch.randn(case["tokens"], case["n"], generator=g, device=DEV)]
    return [x, w, bias]


def prepare(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    s = {"case": case}
    if kind == "roundtrip":
        s["x"] = t[0]
    elif kind == "kv":
        cache = qa.kv_cache_quantizer(case["heads"], case["dim"], case["dtype"], max_seq_len=case["steps"])
        for i in range(case["steps"]):
            cache.append_kv(t[0][i, 0], t[0][i, 1])
        s.update(cache=cache, k=t[0][-1, 0].clone(), v=t[0][-1, 1].clone())
    elif kind == "matmul":
        a, b = t
        if not case["floats"]:
            a = qa.mx_tensor.quantize(a, case["dtype"], case["block"])
            b = qa.mx_tensor.quantize(b, case["dtype"], case["block"])
        s.update(a=a, b=b)
    elif kind in ("linear", "mlp"):
        if kind == "linear":
            model = qa.to_mx(nn.Sequential(_float_linear(t[1])), case["dtype"])
        else:
            model = qa.to_mx(nn.Sequential(_float_linear(t[1]), nn.SiLU(), _float_linear(t[2])), case["dtype"])
        s.update(model=model, x=t[0])
        if case["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.no_grad(), torch.cuda.stream(side):
                model(s["x"])  # the layers lay their weights out, the stream gets its workspace
                graph = torch.cuda.CUDAGraph()
                with torch.cuda.graph(graph, stream=side):
                    s["y"] = model(s["x"])
            torch.cuda.current_stream().wait_stream(side)
            s.update(graph=graph, side=side)
    elif kind == "dynamic":
        s["layer"] = qa.mx_dynamic_linear.from_linear(_float_linear(t[1], t[2]), weight_dtype=case["dtype"])
        s.update(x=t[0].requires_grad_(True), grad=t[3])
    else:
        s.update(x=t[0], w=qa.mx_tensor.quantize(t[1], "int8d", 128), bias=t[2])
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "roundtrip":
        seed = SEED_H if case["dtype"].endswith("h") else None
        q = qa.mx_tensor.quantize(s["x"], case["dtype"], case["block"], seed=seed)
        return q.packed, q.mx_scales, q.dequantize()
    if kind == "kv":
        s["cache"].append_kv(s["k"], s["v"])
        return s["cache"].get()
    if kind == "matmul":
        c = qa.mx_matmul(s["a"], s["b"], case["dtype"], case["block"]) if case["floats"] else s["a"] @ s["b"]
        return c.packed, c.mx_scales
    if kind in ("linear", "mlp"):
        if case["graph"]:
            s["graph"].replay()
            return s["y"]
        with torch.no_grad():
            return s["model"](s["x"])
    if kind == "dynamic":
        y = s["layer"](s["x"])
        (gx,) = torch.autograd.grad(y, s["x"], s["grad"])
        return y.detach(), gx
    return qa.fused_int8_linear(qa.dynamic_quantize(s["x"], "int8d", "per_token"), s["w"], s["bias"])


# ---------------------------------------------------------------- what a pass cannot do without
def _code_bytes(dtype, n):
    bits = int("".join(c for c in dtype if c.isdigit()))
    return n * bits / 8 + n / 128 * 4


def _src_bytes(src):
    return 4 if src == "fp32" else 2


def work(case):
    kind = case["kind"]
    if kind == "roundtrip":
        n = case["rows"] * case["cols"]
        flops = n * 2 * math.log2(case["cols"]) if case["dtype"].endswith("h") else 0
        return {"bytes": n * _src_bytes(case["src"]) + _code_bytes(case["dtype"], n) + 4 * n, "flops": flops}
    if kind == "kv":
        step = 2 * case["batch"] * case["heads"] * case["dim"]
        return {"bytes": step * _src_bytes(case["src"]) + case["steps"] * (_code_bytes(case["dtype"], step) + 4 * step),
                "flops": 0}
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        read = 4 * (m * k + k * n) if case["floats"] else _code_bytes(case["dtype"], m * k + k * n)
        out = {"int8d": "int16d", "int4d": "int8d"}[case["dtype"]]
        return {"bytes": read + _code_bytes(out, m * n), "flops": 2 * m * k * n}
    if kind == "mlp":
        t, d, f = case["tokens"], case["d"], case["f"]
        return {"bytes": _code_bytes(case["dtype"], 2 * d * f) + t * d * (_src_bytes(case["src"]) + 4),
                "flops": 4 * t * d * f}
    t, k, n = case["tokens"], case["k"], case["n"]
    if kind == "linear":
        return {"bytes": _code_bytes(case["dtype"], k * n) + t * k * _src_bytes(case["src"]) + 4 * t * n,
                "flops": 2 * t * k * n}
    if kind == "dynamic":
        return {"bytes": _code_bytes(case["dtype"], k * n) + 2 * t * k * _src_bytes(case["src"]) + 8 * t * n,
                "flops": 4 * t * k * n}
    return {"bytes": _code_bytes("int8d", k * n) + t * k * _src_bytes(case["src"]) + 4 * t * n, "flops": 2 * t * k * n}


def tolerance(case):
    # About four times the measured distance from the 64-bit values:
    #   1.2e-6   32-bit sums of up to 8192 terms;
    #   2.7e-5 a layer (6e-5 for two)   int4 weights at up to 16 rows, whose
    #            codes enter the products as 16-bit subnormals with an offset;
    #   1.7e-3, 2.1e-4   an input gradient rounded to bf16, fp16.
    kind = case["kind"]
    if kind in ("roundtrip", "kv", "matmul"):
        return "exact"
    rel = 5e-6
    if kind != "int8" and case["dtype"] == "int4d" and case["tokens"] <= 16:
        rel = 2.4e-4
    if kind == "dynamic":
        rel = max(rel, {"fp32": 0.0, "bf16": 7e-3, "fp16": 9e-4}[case["src"]])
    return {"rel": rel}


# ---------------------------------------------------------------- the same values in 64 bits
# Codes and scales are whole numbers and 32-bit values of a stated rule, so
# they are made with that rule; what is computed from them is in 64 bits.
def _int_codes(x, bits, block):
    """Base integer rule: scale = RN(1 / RN(RN(1 / absmax) * q)), code = round(x * that inverse)."""
    flat = F.pad(x.float().reshape(-1), (0, -x.numel() % block)).view(-1, block)
    q = float((1 << (bits - 1)) - 1)
    inv = flat.abs().amax(1).clamp(min=1e-12).reciprocal() * q
    return (flat * inv[:, None]).clamp(-q, q).round().double(), inv.reciprocal().double()


def _vector_codes(x, bits, block):
    """Vector rule: scale = absmax / q, code = round(x / scale)."""
    flat = F.pad(x.float().reshape(-1), (0, -x.numel() % block)).view(-1, block)
    q = torch.tensor(float((1 << (bits - 1)) - 1), device=x.device)
    s = flat.abs().amax(1).clamp(min=1e-12) / q
    return (flat / s[:, None]).clamp(-q, q).round().double(), s.double()


def _grid(bits):
    if bits == 4:
        pos = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0])
    else:
        pos = torch.tensor([m / 8 * 2.0 ** -6 if e == 0 else (1 + m / 8) * 2.0 ** (e - 7 if e < 15 else 8)
                            for e in range(16) for m in range(8)])
    pos = pos / pos.max()
    return torch.cat([-pos.flip(0), pos]).sort().values


def _dequantized(x, dtype, block):
    """Value and scales of x after packing with a base format, 64-bit products of codes and scales."""
    bits = int("".join(c for c in dtype if c.isdigit()))
    if dtype.startswith("float"):
        grid = _grid(bits).to(x.device)
        flat = F.pad(x.float().reshape(-1), (0, -x.numel() % block)).view(-1, block)
        s = flat.abs().amax(1).clamp(min=1e-12)
        idx = torch.bucketize(flat / s[:, None], (grid[:-1] + grid[1:]) * 0.5)
        c, s = grid[idx].double(), s.double()
    elif "v" in dtype:
        c, s = _vector_codes(x, bits, block)
    else:
        c, s = _int_codes(x, bits, block)
    return (c * s[:, None]).reshape(-1)[:x.numel()].view(x.shape), s


def _walsh(x):
    """Walsh-Hadamard transform of the rows, widest butterflies first, over the root of the length."""
    d = x.shape[-1]
    h, step = x, d
    while step > 1:
        step //= 2
        h = h.reshape(-1, d // (2 * step), 2, step)
        h = torch.stack([h[:, :, 0] + h[:, :, 1], h[:, :, 0] - h[:, :, 1]], 2)
    return h.reshape(-1, d) / torch.tensor(math.sqrt(d), dtype=x.dtype, device=x.device)


def exact(case, seed):
    kind = case["kind"]
    t = _inputs(case, seed)
    if kind == "roundtrip":
        x, dtype = t[0], case["dtype"]
        if not dtype.endswith("h"):
            y, s = _dequantized(x, dtype, case["block"])
            return None, s, y
        signs = torch.randint(0, 2, (case["cols"],), generator=torch.Generator().manual_seed(SEED_H)).to(DEV) * 2 - 1
        y, s = _dequantized(_walsh(x.float() * signs), dtype[:-1], case["block"])
        return None, s, (_walsh(y) * signs).view(x.shape)
    if kind == "kv":
        h, d = case["heads"], case["dim"]
        out = []
        for i in range(2):
            x = t[0][1:, i].float().reshape(case["steps"], -1, d)
            low = x.amin(-1, keepdim=True) if i else torch.zeros_like(x[..., :1])
            y = _dequantized(x - low, case["dtype"], d)[0] + low.double()
            out.append(y.permute(1, 0, 2).reshape(-1, h, case["steps"], d))
        return tuple(out)
    if kind == "matmul":
        m, k, n, block = case["m"], case["k"], case["n"], case["block"]
        bits = int(case["dtype"][3])
        ca, sa = _int_codes(t[0], bits, block)
        cb, sb = _int_codes(t[1], bits, block)
        ca, cb = ca.reshape(-1)[:m * k].view(m, k), cb.reshape(-1)[:k * n].view(k, n)
        kb = -(-k // block)
        # B's scales are read as one per K block and column, and either
        # operand's as ones where their number does not fit that reading
        sa = sa.view(m, kb) if sa.numel() == m * kb else torch.ones(m, kb, dtype=torch.float64, device=DEV)
        sb = sb.view(kb, n) if sb.numel() == kb * n else torch.ones(kb, n, dtype=torch.float64, device=DEV)
        c = torch.zeros(m, n, dtype=torch.float64, device=DEV)
        for i in range(kb):
            p = ca[:, i * block:(i + 1) * block].contiguous() @ cb[i * block:(i + 1) * block].contiguous()
            c += p * sa[:, i, None] * sb[i]
        q = float((1 << (2 * bits - 1)) - 1)
        c = F.pad(c.reshape(-1), (0, -c.numel() % block)).view(-1, block)
        return None, c.abs().amax(1).clamp(min=1e-12) / q
    if kind in ("linear", "mlp"):
        y = t[0].double()
        for i, w in enumerate(t[1:]):
            y = F.silu(y) if i else y
            y = y @ _dequantized(w.t().contiguous(), case["dtype"], 128)[0]
        return y
    x, w, bias = t[:3]
    if kind == "dynamic":
        wd = _dequantized(w, case["dtype"], 128)[0]
        return x.double() @ wd.t().contiguous() + bias.double(), t[3].double() @ wd
    cx, sx = _vector_codes(x, 8, case["k"])
    wd = _dequantized(w, "int8d", 128)[0]
    return (cx * sx[:, None]) @ wd.t().contiguous() + bias.double()
