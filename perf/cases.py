"""The work that a program built on this package has it do, as measurable cases.

Every case is a dict of plain values; its "kind" says which entry points a pass calls:

  chain    one decode step's projections recorded into a graph and replayed: per layer the Q4_K q/k/v triple, o, the
           gate/up dual and the Q6_K down projection, then the Q6_K head
  kquant   one transformer layer of a Q4_K_M mix: q, k, v, o, gate, up in Q4_K and down in Q6_K.  One token uses the
           triple and dual projections, more tokens the token-batched encoders
  q8       transformer layers in Q8_0 through the fused projections (RMSNorm + QKV, gate/up + SiLU); one token adds the
           residual in the o and down projections, more tokens run those two token-batched
  gemv     one matrix of one format against one or more tokens (an LM head, a single projection)
  gemm     prefill GEMM over raw Q4_K / Q8_0 weights, bf16 activations
  dequant  load-time dequantisation of a whole matrix to fp32
  quantize the Q8_0 row quantizer

Weights are raw GGUF blocks with uniform quants and fp16 scales, activations are normal with a few strong channels, as the
residual stream of a language model has.  All of it is made on the GPU from the seed.
"""
from __future__ import annotations

import math

import torch

from edgerunner_amd import (Buffer, Capture, DequantQ4KMKernel, DequantQ6KKernel, DequantQ8_0Kernel, FusedQ8Kernel,
                            GEMVKernel, QuantGEMMKernel, QuantizeQ8RowsKernel, default_context)
from edgerunner_amd._ffi import er_buffer

BLOCK = {"q8_0": (34, 32), "q4_k": (144, 256), "q6_k": (210, 256)}
EPS = 1e-5
# hidden width, q rows, kv rows, ffn width
SMALL = {"hidden": 1024, "q": 2048, "kv": 1024, "ffn": 3072}      # a 0.6B model's layer
LARGE = {"hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336}     # an 8B model's layer


def listed():
    return [
        # a whole decode step of a 28-layer 0.6B model: 113 small launches, bound by their latency
        {"name": "decode_step_0.6b", "kind": "chain", "layers": 28, "vocab": 151936, **SMALL},
        # decode of the same model size in Q8_0, eight layers called one launch after the other, as a plain loop does
        {"name": "decode_q8_8_layers_0.6b", "kind": "q8", "layers": 8, "tokens": 1, **SMALL},
        # one layer of an 8B model in decode: the bandwidth-bound case
        {"name": "decode_layer_8b", "kind": "kquant", "tokens": 1, **LARGE},
        # the logits of an 8B model's head
        {"name": "head_q6k_128256", "kind": "gemv", "fmt": "q6_k", "tokens": 1, "M": 128256, "K": 4096},
        # checking a draft of five tokens (or five users) in one pass over an 8B layer
        {"name": "verify_5_layer_8b", "kind": "kquant", "tokens": 5, **LARGE},
        # a short prompt through one layer of the 0.6B model, token-batched
        {"name": "prompt_32_layer_0.6b", "kind": "kquant", "tokens": 32, **SMALL},
        # an odd-length prompt through one 8B layer in Q8_0: the token-batched fused projections are the fp32 prefill
        {"name": "prompt_77_q8_layer_8b", "kind": "q8", "layers": 1, "tokens": 77, **LARGE},
        # prefill of a 512-token chunk, and of a short ragged one, and of a long prompt
        {"name": "prefill_512_q4k", "kind": "gemm", "fmt": "q4_k", "tokens": 512, "N": 14336, "K": 4096},
        {"name": "prefill_100_q8", "kind": "gemm", "fmt": "q8_0", "tokens": 100, "N": 4096, "K": 4096},
        {"name": "prefill_4096_q4k", "kind": "gemm", "fmt": "q4_k", "tokens": 4096, "N": 14336, "K": 4096},
        # loading: a feed-forward matrix widened to fp32
        {"name": "dequant_q6k", "kind": "dequant", "fmt": "q6_k", "M": 14336, "K": 4096},
        # fp32 rows written as Q8_0 blocks
        {"name": "quantize_2048", "kind": "quantize", "rows": 2048, "K": 4096},
    ]


def _log(rng, lo, hi, step=1):
    """An integer multiple of `step` from [lo, hi], its logarithm spread evenly."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi // step, max(-(-lo // step), round(v / step))) * step


MOST = 1.6e10  # weights times tokens of a drawn token-batched pass: the listed 77-token prompt's


def draw(rng):
    kind = rng.choice(["kquant", "kquant", "q8", "gemv", "gemv", "gemm", "gemm", "dequant", "quantize", "chain"])
    if kind == "gemm":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q8_0"]), "tokens": _log(rng, 16, 4096),
                "N": _log(rng, 1024, 14336, 8), "K": _log(rng, 1024, 4096, 256)}
    if kind == "gemv":
        fmt, M, K = rng.choice(["q4_k", "q6_k", "q8_0"]), _log(rng, 2048, 32768, 4), _log(rng, 1024, 14336, 256)
        return {"kind": kind, "fmt": fmt, "tokens": min(rng.choice([1, 1, _log(rng, 2, 96)]), int(MOST / (M * K))), "M": M, "K": K}
    if kind == "dequant":
        return {"kind": kind, "fmt": rng.choice(["q4_k", "q6_k", "q8_0"]), "M": _log(rng, 2048, 28672), "K": 256 * rng.randint(4, 20)}
    if kind == "quantize":
        return {"kind": kind, "rows": _log(rng, 64, 8192), "K": 64 * rng.randint(16, 128)}
    dims = {"hidden": 256 * rng.randint(4, 20), "kv": 128 * rng.randint(4, 10), "ffn": 256 * rng.randint(12, 56)}
    dims["q"] = rng.choice([dims["hidden"], 2048])
    if kind == "chain":
        return {"kind": kind, "layers": rng.randint(2, 12), "vocab": 4 * rng.randint(8000, 40000), "hidden": 1024,
                "q": 2048, "kv": 1024, "ffn": 256 * rng.randint(8, 16)}
    weights = sum(M * K for M, K in _layer_shapes(dims).values())
    tokens = min(rng.choice([1, _log(rng, 2, 8), _log(rng, 8, 96)]), int(MOST / weights))
    if kind == "kquant":
        return {"kind": kind, "tokens": tokens, **dims}
    return {"kind": kind, "layers": 1, "tokens": tokens, **dims}


# ---------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _weights(fmt, M, K, g):
    """Raw GGUF blocks [M, K / block, bytes]: uniform quants, fp16 scales of both signs' usual size."""
    nbytes, per = BLOCK[fmt]
    n = M * (K // per)
    w = torch.randint(0, 256, (n, nbytes), dtype=torch.uint8, device="cuda", generator=g)

    def scale(s):
        return ((torch.rand(n, device="cuda", generator=g) + 0.25) * s).half().view(torch.uint8).view(n, 2)
    if fmt == "q8_0":
        w[:, :2] = scale(0.001)
    elif fmt == "q4_k":
        w[:, 0:2] = scale(0.0005)
        w[:, 2:4] = scale(0.004)
    else:
        w[:, 208:210] = scale(0.0001)
    return w


def _x(T, K, g):
    x = torch.randn(T, K, device="cuda", generator=g)
    strong = torch.rand(K, device="cuda", generator=g) < 0.005
    return torch.where(strong, x * 12.0, x).contiguous()


def _buf(t, ctx):
    return Buffer(ctx, er_buffer(t.data_ptr(), t.numel() * t.element_size()), owned=False)


class _State:
    """Tensors by name, the Buffer of each, and the kernels a program keeps."""

    def __init__(self, case):
        self.case, self.ctx, self.t, self.b = case, default_context(), {}, {}

    def add(self, name, tensor):
        self.t[name] = tensor
        self.b[name] = _buf(tensor, self.ctx)

    def out(self, name, *shape, dtype=torch.float32):
        self.add(name, torch.empty(*shape, dtype=dtype, device="cuda"))


def _layer_shapes(c):
    return {"q": (c["q"], c["hidden"]), "k": (c["kv"], c["hidden"]), "v": (c["kv"], c["hidden"]), "o": (c["hidden"], c["q"]),
            "gate": (c["ffn"], c["hidden"]), "up": (c["ffn"], c["hidden"]), "down": (c["hidden"], c["ffn"])}


def _layer_fmt(c, name):
    return "q8_0" if c["kind"] == "q8" else "q6_k" if name == "down" else "q4_k"


def _inputs(case, seed):
    """The input tensors of a case by name, from the seed alone (prepare() and exact() share it)."""
    c, g, t = case, _generator(seed), {}
    kind = c["kind"]
    if kind in ("chain", "kquant", "q8"):
        T = c.get("tokens", 1)
        for l in range(c.get("layers", 1)):
            for n, (M, K) in _layer_shapes(c).items():
                t[f"w{l}.{n}"] = _weights(_layer_fmt(c, n), M, K, g)
        if kind == "chain":
            t["w.head"] = _weights("q6_k", c["vocab"], c["hidden"], g)
        t["x.h"], t["x.a"], t["x.f"] = _x(T, c["hidden"], g), _x(T, c["q"], g), _x(T, c["ffn"], g)
        if kind == "q8":
            t["norm"] = torch.rand(c["hidden"], device="cuda", generator=g) + 0.5
            if T == 1:
                t["res"] = _x(1, c["hidden"], g)
    elif kind == "gemv":
        t["w"], t["x"] = _weights(c["fmt"], c["M"], c["K"], g), _x(c["tokens"], c["K"], g)
    elif kind == "gemm":
        t["w"], t["x"] = _weights(c["fmt"], c["N"], c["K"], g), _x(c["tokens"], c["K"], g).bfloat16()
    elif kind == "dequant":
        t["w"] = _weights(c["fmt"], c["M"], c["K"], g)
    else:
        t["x"] = _x(c["rows"], c["K"], g)
    return t


def prepare(case, seed):
    s = _State(case)
    for name, tensor in _inputs(case, seed).items():
        s.add(name, tensor)
    c, kind, ctx = case, case["kind"], s.ctx
    if kind in ("chain", "kquant", "q8"):
        s.gemv, s.fused = GEMVKernel(ctx), FusedQ8Kernel(ctx)
        T, shapes = c.get("tokens", 1), _layer_shapes(c)
        names = ("q", "k", "v", "o", "act", "down") if kind == "q8" else tuple(shapes)
        rows = {n: c["ffn"] if n == "act" else shapes[n][0] for n in names}
        if kind == "chain":  # one output tensor for all layers, as 28 x 7 of them would be
            s.add("y", torch.empty(c["layers"], sum(rows.values()), device="cuda"))
            s.out("logits", c["vocab"])
            for l in range(c["layers"]):
                at = 0
                for n in names:
                    s.b[f"y{l}.{n}"] = _buf(s.t["y"][l, at:at + rows[n]], ctx)
                    at += rows[n]
            torch.cuda.synchronize()
            s.stream = ctx.stream()
            with Capture(ctx, s.stream) as cap:
                for l in range(c["layers"]):
                    _decode_layer(s, l, s.stream)
                s.gemv.encodeQ6KWeights(s.stream, s.b["w.head"], s.b["x.h"], s.b["logits"], c["vocab"], c["hidden"])
            s.graph = cap.graph
        else:
            for l in range(c.get("layers", 1)):
                for n in names:
                    half = kind == "q8" and n == "v" and T == 1  # fp16 V goes to the KV cache in decode
                    s.out(f"y{l}.{n}", T, rows[n], dtype=torch.float16 if half else torch.float32)
    elif kind == "gemv":
        s.gemv = GEMVKernel(ctx)
        s.out("y", c["tokens"], c["M"])
    elif kind == "gemm":
        s.gemm = QuantGEMMKernel(ctx)
        s.out("y", c["tokens"], c["N"])
    elif kind == "dequant":
        s.kernel = {"q8_0": DequantQ8_0Kernel, "q4_k": DequantQ4KMKernel, "q6_k": DequantQ6KKernel}[c["fmt"]](ctx)
        s.out("y", c["M"], c["K"])
    else:
        s.kernel = QuantizeQ8RowsKernel(ctx)
        s.out("y", c["rows"], c["K"] // 32 * 34, dtype=torch.uint8)
    return s


# ---------------------------------------------------------------- one pass

def _decode_layer(s, l, stream):
    """One token through a Q4_K / Q6_K layer: triple, o, dual, down."""
    c, b, g = s.case, s.b, s.gemv
    g.encodeQ4KWeightsTriple(stream, b[f"w{l}.q"], b[f"w{l}.k"], b[f"w{l}.v"], b["x.h"], b[f"y{l}.q"], b[f"y{l}.k"],
                             b[f"y{l}.v"], c["q"], c["kv"], c["kv"], c["hidden"])
    g.encodeQ4KWeights(stream, b[f"w{l}.o"], b["x.a"], b[f"y{l}.o"], c["hidden"], c["q"])
    g.encodeQ4KWeightsDual(stream, b[f"w{l}.gate"], b[f"w{l}.up"], b["x.h"], b[f"y{l}.gate"], b[f"y{l}.up"], c["ffn"],
                           c["hidden"])
    g.encodeQ6KWeights(stream, b[f"w{l}.down"], b["x.f"], b[f"y{l}.down"], c["hidden"], c["ffn"])


def _batched_layer(s):
    c, b, g, T = s.case, s.b, s.gemv, s.case["tokens"]
    for n, (M, K) in _layer_shapes(c).items():
        x = b["x.a" if n == "o" else "x.f" if n == "down" else "x.h"]
        enc = g.encodeBatchedQ6KWeights if n == "down" else g.encodeBatchedQ4KWeights
        enc(None, b[f"w0.{n}"], x, b[f"y0.{n}"], T, M, K)


def _q8_layer(s, l):
    c, b, f, T = s.case, s.b, s.fused, s.case["tokens"]
    qkv = f.encodeFusedQKV if T == 1 else f.encodeFusedQKVTurbo
    qkv(None, b[f"w{l}.q"], b[f"w{l}.k"], b[f"w{l}.v"], b["x.h"], b[f"y{l}.q"], b[f"y{l}.k"], b[f"y{l}.v"], b["norm"],
        c["q"], c["kv"], c["hidden"], T, EPS)
    if T == 1:
        f.encodeGEMVAdd(None, b[f"w{l}.o"], b["x.a"], b["res"], b[f"y{l}.o"], c["hidden"], c["q"])
    else:
        s.gemv.encodeBatchedQ8_0Weights(None, b[f"w{l}.o"], b["x.a"], b[f"y{l}.o"], T, c["hidden"], c["q"])
    f.encodeFusedGateUpSilu(None, b[f"w{l}.gate"], b[f"w{l}.up"], b["x.h"], b[f"y{l}.act"], b["norm"], c["ffn"],
                            c["hidden"], T, EPS)
    if T == 1:
        f.encodeGEMVAdd(None, b[f"w{l}.down"], b["x.f"], b["res"], b[f"y{l}.down"], c["hidden"], c["ffn"])
    else:
        s.gemv.encodeBatchedQ8_0Weights(None, b[f"w{l}.down"], b["x.f"], b[f"y{l}.down"], T, c["hidden"], c["ffn"])


def run(s):
    c, kind, b = s.case, s.case["kind"], s.b
    if kind == "chain":
        s.graph.launch(None)
        return {"y": s.t["y"], "logits": s.t["logits"]}
    if kind == "kquant":
        if c["tokens"] == 1:
            _decode_layer(s, 0, None)
        else:
            _batched_layer(s)
    elif kind == "q8":
        for l in range(c["layers"]):
            _q8_layer(s, l)
    elif kind == "gemv":
        name = {"q4_k": "Q4K", "q6_k": "Q6K", "q8_0": "Q8_0"}[c["fmt"]]
        if c["tokens"] == 1:
            getattr(s.gemv, f"encode{name}Weights")(None, b["w"], b["x"], b["y"], c["M"], c["K"])
        else:
            getattr(s.gemv, f"encodeBatched{name}Weights")(None, b["w"], b["x"], b["y"], c["tokens"], c["M"], c["K"])
    elif kind == "gemm":
        enc = s.gemm.encodeQ4K if c["fmt"] == "q4_k" else s.gemm.encodeQ8_0
        enc(None, b["w"], b["x"], b["y"], c["tokens"], c["N"], c["K"])
    elif kind == "dequant":
        s.kernel.encode(None, b["w"], s.t["w"].shape[0], b["y"])
    else:
        s.kernel.encode(None, b["x"], b["y"], c["rows"], c["K"], 0, c["K"] // 32)
    return {n: t for n, t in s.t.items() if n.startswith("y")}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    c, kind = case, case["kind"]
    if kind in ("chain", "kquant", "q8"):
        T, nbytes, flops = c.get("tokens", 1), 0, 0
        for n, (M, K) in _layer_shapes(c).items():
            bb, per = BLOCK[_layer_fmt(c, n)]
            fused_up = kind == "q8" and n == "up"  # gate and up leave one activated vector
            nbytes += M * (K // per) * bb + (0 if fused_up else 4 * T * M)
            flops += 2 * T * M * K
        L = c.get("layers", 1)
        nbytes, flops = nbytes * L, flops * L
        nbytes += 4 * T * (c["hidden"] + c["q"] + c["ffn"])
        if kind == "chain":
            nbytes += c["vocab"] * (c["hidden"] // 256) * 210 + 4 * c["vocab"]
            flops += 2 * c["vocab"] * c["hidden"]
        return {"bytes": nbytes, "flops": flops}
    if kind == "gemv":
        bb, per = BLOCK[c["fmt"]]
        return {"bytes": c["M"] * (c["K"] // per) * bb + 4 * c["tokens"] * (c["M"] + c["K"]),
                "flops": 2 * c["tokens"] * c["M"] * c["K"]}
    if kind == "gemm":
        bb, per = BLOCK[c["fmt"]]
        return {"bytes": c["N"] * (c["K"] // per) * bb + c["tokens"] * (2 * c["K"] + 4 * c["N"]),
                "flops": 2 * c["tokens"] * c["N"] * c["K"]}
    if kind == "dequant":
        bb, per = BLOCK[c["fmt"]]
        return {"bytes": c["M"] * (c["K"] // per) * bb + 4 * c["M"] * c["K"], "flops": c["M"] * c["K"]}
    return {"bytes": c["rows"] * c["K"] * 4 + c["rows"] * (c["K"] // 32) * 34, "flops": 2 * c["rows"] * c["K"]}


def tolerance(case):
    if case["kind"] in ("dequant", "quantize"):
        return "exact"  # every dequantised value is exact in fp32; quantised blocks are bytes
    if case["kind"] == "gemm":
        return {"rel": 5e-3}  # weights rounded to bf16 (8 bits), fp32 sums: 1.2e-3 from the 64-bit product
    if case["kind"] == "q8" and case["tokens"] == 1:
        return {"rel": 2e-4}  # V is stored in fp16, where a neighbouring value is 2^-11 away
    return {"rel": 4e-6}  # fp32 activations with 22 bits or more, exact products, fp32 sums


# ---------------------------------------------------------------- the same in 64 bits

def _dequant64(w, fmt, M, K):
    d = w[:, :2].contiguous().view(torch.float16).double()
    if fmt == "q8_0":
        v = w[:, 2:].contiguous().view(torch.int8).double() * d
    elif fmt == "q4_k":
        dmin = w[:, 2:4].contiguous().view(torch.float16).double()
        s = w[:, 4:16].int()
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double()
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()
        qs = w[:, 16:].view(-1, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).double()
        v = (d * sc)[:, :, None] * q - (dmin * mn)[:, :, None]
    else:
        d = w[:, 208:210].contiguous().view(torch.float16).double()
        ql, qh = w[:, :128].view(-1, 2, 2, 32).int(), w[:, 128:192].view(-1, 2, 32).int()
        sc = w[:, 192:208].contiguous().view(torch.int8).view(-1, 2, 4, 2).double()
        parts = [((ql[:, :, m & 1] >> (4 * (m >> 1))) & 15) | (((qh >> (2 * m)) & 3) << 4) for m in range(4)]
        q = torch.stack(parts, 2).sub(32).double().view(-1, 2, 4, 2, 16)  # half, quarter, 16s
        v = d[:, :, None, None, None] * sc[..., None] * q
    return v.reshape(M, K)


def _mul64(w, fmt, M, K, x):
    """x [T, K] times the dequantised rows, in pieces of rows that fit easily."""
    per = K // BLOCK[fmt][1]
    x, out, step = x.double(), [], max(1, (1 << 26) // K)
    for r in range(0, M, step):
        m = min(step, M - r)
        out.append(x @ _dequant64(w[r * per:(r + m) * per], fmt, m, K).T.contiguous())
    return torch.cat(out, 1)


def exact(case, seed):
    if case["kind"] == "quantize":
        return None  # bytes
    c, kind, t = case, case["kind"], _inputs(case, seed)
    if kind == "dequant":
        return {"y": _dequant64(t["w"], c["fmt"], c["M"], c["K"])}
    if kind == "gemv":
        return {"y": _mul64(t["w"], c["fmt"], c["M"], c["K"], t["x"])}
    if kind == "gemm":
        return {"y": _mul64(t["w"], c["fmt"], c["N"], c["K"], t["x"])}
    shapes = _layer_shapes(c)

    def proj(l, n, x):
        return _mul64(t[f"w{l}.{n}"], _layer_fmt(c, n), *shapes[n], x)
    h, a, f = t["x.h"], t["x.a"], t["x.f"]
    if kind == "kquant":
        return {f"y0.{n}": proj(0, n, a if n == "o" else f if n == "down" else h) for n in shapes}
    if kind == "chain":
        rows = [torch.cat([proj(l, n, a if n == "o" else f if n == "down" else h) for n in shapes], 1)
                for l in range(c["layers"])]
        return {"y": torch.cat(rows, 0), "logits": _mul64(t["w.head"], "q6_k", c["vocab"], c["hidden"], h)[0]}
    h = h.double()
    h = h / torch.sqrt((h * h).mean(1, keepdim=True) + EPS) * t["norm"].double()
    res = t["res"].double() if "res" in t else 0.0
    out = {}
    for l in range(c["layers"]):
        for n in ("q", "k", "v"):
            out[f"y{l}.{n}"] = proj(l, n, h)
        out[f"y{l}.o"] = proj(l, "o", a) + res
        g = proj(l, "gate", h)
        out[f"y{l}.act"] = g / (1.0 + torch.exp(-g)) * proj(l, "up", h)
        out[f"y{l}.down"] = proj(l, "down", f) + res
    return out
