"""What a serving program has this library do, as a list of cases that can be timed.

A case is a dict of plain values; `prepare` makes the program's weights, buffers and handles for it from a seed, `run`
is one pass through the public entry points.  Kinds:

  linear  one (possibly stacked) block linear over a batch of rows: PackedShards.forward, or the torch op that the
          vLLM linear method calls
  layer   the block linears of decoder layers in order, with the residual adds, norms and SiLU product between them;
          eagerly or as the HIP graph that a decode loop captures once and replays
  ends    the two ends of a serving step: the 4-bit token embedding of its input rows and the 8-bit output head over
          the rows that want logits
  load    one stacked linear brought up from the packed file's tensors in host memory: the cost of a model's start

The layer shapes, formats and row counts are those of bench.py and the tests, or generic.
"""

from __future__ import annotations

import math

import torch

from quantexperiments_amd.kernels import (PackedLinear, addnorm, linear_small, linear_small_from, linear_small_silu,
                                          silu_mul)
from quantexperiments_amd.masks import seeded_perms
from quantexperiments_amd.vllm_ext import core

SMALL = 32          # most rows of a decode step


# ------------------------------------------------------------------ the cases

def _linear(name, outs, C, d, bits, rows, **kw):
    return {"name": name, "kind": "linear", "outs": outs, "C": C, "d": d, "bits": bits, "G": 1, "M": 1, "rows": rows,
            "dtype": "bf16", "tags": "uniform", "large": "fused", "op": False, **kw}


def _layer(name, hidden, kv, inter, d, bits, rows, **kw):
    return {"name": name, "kind": "layer", "hidden": hidden, "kv": kv, "inter": inter, "d": d, "bits": bits, "G": 1,
            "M": 1, "rows": rows, "dtype": "bf16", "layers": 1, "graph": False, **kw}


def listed():
    return [
        # one token of a small model, eagerly through the op of the vLLM linear method: latency and launches
        _linear("one_small_row", "4864", 896, 4, 8, 1, op=True),
        # batch-1 decode of a 7B-shaped layer at 2 bits per weight, captured as a decode loop captures it
        _layer("decode_k65536_1row", 3584, 512, 18944, 8, 16, 1, graph=True),
        # batch-1 q|k|v of a 27B-class layer with 16 column orders and uneven codeword popularity, eagerly
        _linear("decode_orders_1row", "5120,1024,1024", 5120, 8, 16, 1, M=16, tags="zipf"),
        # a decode batch of 8 sequences at 3 bits per weight, two layers in one graph
        _layer("decode_k4096_8rows", 3584, 512, 18944, 4, 12, 8, layers=2, graph=True),
        # a decode batch run without a graph, several codebooks per matrix, fp16 activations
        _layer("decode_4books_4rows", 5120, 1024, 17408, 4, 12, 4, G=4, dtype="f16"),
        # a short prompt or a batch of drafted tokens: more rows than a decode step, far fewer than a prefill
        _layer("short_prompt_77rows", 3584, 512, 18944, 4, 10, 77),
        # a ragged chunk of a chunked prefill on the gate|up projection, fp16
        _linear("chunk_333rows", "18944,18944", 3584, 8, 16, 333, dtype="f16"),
        # prefill of a long prompt: gate|up at 2048 rows
        _linear("prefill_k65536_2048rows", "18944,18944", 3584, 8, 16, 2048),
        # prefill with column orders through the decode-to-dense route
        _linear("prefill_orders_1024rows", "5120,1024,1024", 5120, 8, 16, 1024, M=16, large="dequant"),
        # prefill of a whole layer with its elementwise neighbours
        _layer("prefill_k4096_2048rows", 3584, 512, 18944, 4, 12, 2048),
        # ends of a mixed serving step: 2048 input tokens, 16 sequences that want logits
        {"name": "ends_2048in_16out", "kind": "ends", "vocab": 152064, "C": 3584, "rows_in": 2048, "rows_out": 16,
         "dtype": "bf16"},
        # start of a model: an attention input projection from the file's tensors
        {"name": "load_k65536", "kind": "load", "outs": "3584,512,512", "C": 3584, "d": 8, "bits": 16, "G": 1, "M": 1,
         "rows": 1, "dtype": "bf16", "tags": "uniform"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi, step, d):
    """A row length: mostly a multiple of 64, now and then any multiple of `step` chunks."""
    u = 64 if rng.random() < 0.85 else step * d
    return max(u, _log(rng, lo, hi) // u * u)


# the formats of bench.py, the tests and the packed files: (chunk length, tag bits)
_FORMATS = ((8, 16), (8, 16), (4, 12), (4, 12), (4, 10), (4, 8))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "layer", "layer", "ends", "load"))
    dtype = rng.choice(("bf16", "bf16", "f16"))
    if kind == "ends":
        return {"kind": "ends", "vocab": _log(rng, 8000, 152064), "C": _width(rng, 512, 3584, 32, 1),
                "rows_in": _log(rng, 1, 2048), "rows_out": _log(rng, 1, 64), "dtype": dtype}
    if kind == "load":
        d, bits = rng.choice(((8, 16), (8, 16), (4, 12)))
        return {"kind": "load", "outs": str(_log(rng, 256, 4096)), "C": _width(rng, 512, 3584, 4, d), "d": d, "bits": bits,
                "G": 1, "M": rng.choice((1, 1, 16)) if d == 8 else 1, "rows": rng.choice((1, 2, 4)), "dtype": dtype,
                "tags": "uniform"}
    d, bits = rng.choice(_FORMATS)
    G = rng.choice((1, 1, 1, 4)) if d == 4 else 1
    M = rng.choice((1, 1, 16)) if d == 8 else 1
    # decode, between decode and prefill, prefill
    part = rng.choice(("decode", "decode", "middle", "prefill"))
    rows = {"decode": lambda: _log(rng, 1, 32), "middle": lambda: _log(rng, 33, 511), "prefill": lambda: _log(rng, 512, 2048)}[part]()
    if kind == "linear":
        C = _width(rng, 512, 5120, 4, d)
        first = _log(rng, 256, 18944)
        outs = rng.choice((str(first), "%d,%d" % (first, first), "%d,%d,%d" % (first, max(64, first // 4), max(64, first // 4))))
        return _drop_name(_linear("", outs, C, d, bits, rows, G=G, M=M, dtype=dtype,
                                  tags=rng.choice(("uniform", "zipf")) if bits == 16 else "uniform",
                                  large=rng.choice(("fused", "fused", "dequant")), op=rng.random() < 0.25 and first * C < 4 << 20))
    hidden = _width(rng, 512, 3584, 2, d)
    inter = max(64, int(hidden * rng.uniform(2.5, 5.3)) // 64 * 64)
    return _drop_name(_layer("", hidden, max(64, hidden // rng.choice((1, 4, 7)) // 8 * 8), inter, d, bits, rows, G=G, M=M, dtype=dtype,
                             graph=part == "decode" and rng.random() < 0.6, layers=1))


def _drop_name(case):
    del case["name"]
    return case


# ------------------------------------------------------------------ what a program has in hand before the call

_DT = {"bf16": torch.bfloat16, "f16": torch.float16}


def _tensors(case, R, C, gen, host):
    """The packed file's tensors of one matrix (tags, table, row scales, codebook and column-order ids) and its orders."""
    dev, d, bits, G, M = gen.device, case["d"], case["bits"], case["G"], case["M"]
    n = C // d
    W = (n * bits + 31) // 32
    if case.get("tags") == "zipf":                    # codeword popularity 1 / rank, popular codewords scattered
        w = 1.0 / torch.arange(1, (1 << bits) + 1, device=dev, dtype=torch.float64)
        cdf = torch.cumsum(w / w.sum(), 0).float()
        rank = torch.searchsorted(cdf, torch.rand(R, n + n % 2, device=dev, generator=gen)).clamp_(max=(1 << bits) - 1)
        tags = torch.randperm(1 << bits, device=dev, generator=gen)[rank]
        words = (tags[:, ::2] | tags[:, 1::2] << 16).to(torch.int32)
    else:
        words = torch.randint(-2 ** 31, 2 ** 31, (R, W), device=dev, dtype=torch.int64, generator=gen).to(torch.int32)
    used = n * bits - (W - 1) * 32
    if used < 32:
        words[:, -1] &= (1 << used) - 1               # the bits behind a row's last tag are zero in a file
    t = {"words": words, "table": torch.randn(G << bits, d, device=dev, generator=gen).half(),
         "row_scale": (torch.randn(R, device=dev, generator=gen) * 0.005 + 0.02).abs().half(),
         "row_book": torch.randint(0, G, (R,), device=dev, generator=gen).to(torch.uint8) if G > 1 else None,
         "row_mask": torch.randint(0, M, (R,), device=dev, generator=gen).to(torch.uint8) if M > 1 else None}
    cpu = torch.Generator().manual_seed(int(torch.randint(0, 2 ** 31, (1,), device=dev, generator=gen)))
    t["perms"] = seeded_perms(C, M, cpu)
    return {k: v if v is None else v.cpu() if host else v.to(dev) for k, v in t.items()}


def _shards(case, outs, C, gen):
    later = "later" if len(outs) > 1 else True
    rls = [PackedLinear(**_tensors(case, R, C, gen, False), K=1 << case["bits"], d=case["d"], stream=later) for R in outs]
    return core.PackedShards(rls, large=case.get("large", "fused"))


class _Layers:
    """Decoder layers without their attention: every layer takes the attention's output as given."""

    def __init__(self, case, gen):
        H, kv, I, B = case["hidden"], case["kv"], case["inter"], case["rows"]
        dev, dt = gen.device, _DT[case["dtype"]]
        self.layers = [{"qkv": _shards(case, (H, kv, kv), H, gen), "o": _shards(case, (H,), H, gen),
                        "gate_up": _shards(case, (I, I), H, gen), "down": _shards(case, (H,), I, gen),
                        "norm1": (torch.rand(H, device=dev, generator=gen) + 0.5).to(dt),
                        "norm2": (torch.rand(H, device=dev, generator=gen) + 0.5).to(dt)} for _ in range(case["layers"])]
        self.h = torch.randn(B, H, device=dev, generator=gen)
        self.prev = torch.randn(B, H, device=dev, generator=gen).to(dt)
        self.attn = torch.randn(B, H, device=dev, generator=gen).to(dt)
        self.decode = B <= SMALL
        # a program's own activation buffers, one set per layer
        new = lambda n, t=dt: torch.empty(B, n, device=dev, dtype=t)
        self.bufs = [{"x1": new(H), "x2": new(H), "h1": new(H, torch.float32), "h2": new(H, torch.float32),
                      "qkv": new(H + 2 * kv), "o": new(H), "act": new(I), "down": new(H)} for _ in self.layers]

    def step(self):
        h, prev, out = self.h, self.prev, []
        for L, b in zip(self.layers, self.bufs):
            if self.decode:
                linear_small_from(L["qkv"].rls, b["qkv"], b["x1"], h_in=h, add=prev, w=L["norm1"], eps=1e-6, h_out=b["h1"])
                linear_small(L["o"].rls, self.attn, b["o"])
                norm2 = {"h_in": b["h1"], "add": b["o"], "w": L["norm2"], "eps": 1e-6, "h_out": b["h2"], "x_out": b["x2"]}
                if self.attn.shape[0] == 1:
                    linear_small_silu(L["gate_up"].rls, None, b["act"], **norm2)
                else:
                    addnorm(b["h1"], b["o"], L["norm2"], 1e-6, b["x2"], h_out=b["h2"])
                    linear_small_silu(L["gate_up"].rls, b["x2"], b["act"])
                linear_small(L["down"].rls, b["act"], b["down"])
                qkv, o, act, prev = b["qkv"], b["o"], b["act"], b["down"]
            else:
                addnorm(h, prev, L["norm1"], 1e-6, b["x1"], h_out=b["h1"])
                qkv = L["qkv"].forward(b["x1"])
                o = L["o"].forward(self.attn)
                addnorm(b["h1"], o, L["norm2"], 1e-6, b["x2"], h_out=b["h2"])
                gu = L["gate_up"].forward(b["x2"])
                act = silu_mul(gu[:, :b["act"].shape[1]], gu[:, b["act"].shape[1]:], b["act"])
                prev = L["down"].forward(act)
            h = b["h2"]
            out.append({"qkv": qkv, "o": o, "act": act, "down": prev, "h": h})
        return out

    def capture(self):
        self.step()                                   # the library's workspace grows outside the capture
        torch.cuda.synchronize()
        self.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(self.graph):
            self.out = self.step()

    def replay(self):
        self.graph.replay()
        return self.out


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    dt = _DT[case["dtype"]]
    kind = case["kind"]
    if kind == "layer":
        s = _Layers(case, gen)
        if case["graph"]:
            s.capture()
            return s.replay
        return s.step
    if kind == "ends":
        V, C = case["vocab"], case["C"]
        q4 = torch.randint(0, 256, (V, C // 2), device=dev, dtype=torch.uint8, generator=gen)
        q8 = torch.randint(-127, 128, (V, C), device=dev, dtype=torch.int8, generator=gen)
        s4, s8 = ((torch.rand(V, C // 32, device=dev, generator=gen) * 0.002 + 0.0005).half() for _ in range(2))
        embed, head = core.Q4Embedding(q4, s4, dt), core.Q8Head(q8, s8)
        ids = torch.randint(0, V, (case["rows_in"],), device=dev, generator=gen)
        x = torch.randn(case["rows_out"], C, device=dev, generator=gen).to(dt)
        return lambda: {"embed": embed.forward(ids), "logits": head.forward(x)}
    outs, C = [int(r) for r in case["outs"].split(",")], case["C"]
    x = torch.randn(case["rows"], C, device=dev, generator=gen).to(dt)
    if kind == "load":
        files = [_tensors(case, R, C, gen, True) for R in outs]

        def load():
            later = "later" if len(files) > 1 else True
            rls = [PackedLinear(**{k: v if v is None else v.to(dev) for k, v in f.items()}, K=1 << case["bits"], d=case["d"],
                                stream=later) for f in files]
            ps = core.PackedShards(rls)
            return {"dense": ps.dense(), "y": ps.forward(x)}
        return load
    ps = _shards(case, outs, C, gen)
    if case["op"]:
        handle = core.register(ps)
        return lambda: torch.ops.shapequant.linear(x, handle)
    return lambda: ps.forward(x)


def run(state):
    return state()


# ------------------------------------------------------------------ what a pass cannot do without

def _matrix_bytes(case, R, C):
    d, bits, G, M = case["d"], case["bits"], case["G"], case["M"]
    n = R * ((C // d * bits + 31) // 32) * 4 + (G << bits) * d * 2 + R * 2
    return n + (R if G > 1 else 0) + (R + M * C * 4 if M > 1 else 0)


def work(case):
    kind = case["kind"]
    if kind == "ends":
        V, C, n, B = case["vocab"], case["C"], case["rows_in"], case["rows_out"]
        rows = min(n, V)
        return {"bytes": n * 8 + rows * (C // 2 + C // 16) + n * C * 2 + V * (C + C // 16) + B * C * 2 + B * V * 2,
                "flops": 2 * B * V * C}
    B = case["rows"]
    if kind == "layer":
        H, kv, I = case["hidden"], case["kv"], case["inter"]
        stacks = (((H, kv, kv), H), ((H,), H), ((I, I), H), ((H,), I))
        n = sum(_matrix_bytes(case, R, C) for outs, C in stacks for R in outs) + 2 * H * 2
        # in: residual stream, previous output, attention output; out: q|k|v, o, SiLU product, down, residual stream
        n += B * (H * 4 + 2 * H * 2 + (H + 2 * kv + H + I + H) * 2 + H * 4)
        return {"bytes": n * case["layers"], "flops": 2 * B * case["layers"] * sum(sum(outs) * C for outs, C in stacks)}
    outs, C = [int(r) for r in case["outs"].split(",")], case["C"]
    n = sum(_matrix_bytes(case, R, C) for R in outs) + B * C * 2 + B * sum(outs) * 2
    if kind == "load":
        n += sum(outs) * C * 2
    return {"bytes": n, "flops": 2 * B * sum(outs) * C}


def tolerance(case):
    """Inputs, weights and outputs of 16 bits with 32-bit sums.  A layer rounds its activations to 16 bits between its
    products, so what one rounding decided differently passes through the next product."""
    unit = 2.0 ** -8 if case["dtype"] == "bf16" else 2.0 ** -11
    return {"rel": (2.0 if case["kind"] == "layer" else 1.0) * unit}
