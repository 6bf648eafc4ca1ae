"""Timed cases of the library's public entry points (include/g4.h).

Sizes are those of the Gemma-4-E2B shape the library runs: hidden width 1536,
FFN 6144 / 12288, 8 query heads on one key/value head of 256 (sliding window
512) or 512 (global) channels, passes of 1 to 512 tokens.  Five kinds:

  generate  a whole conversation turn through g4_forward / g4_logits: the
            prompt in passes of at most 512 tokens from position 0 and the
            logits of its last row, then `steps` one-token passes with their
            logits (the reply, its tokens given)
  matmul    one W8A8 product, g4_matmul_int8 (1 row: decode; 2-8: a few
            tokens checked at once; more: prompts up to a whole chunk)
  attend    attention of n tokens over a KV ring, g4_attend
  layer     the attention block: g4_rmsnorm, then g4_attention_layer
  ffn       the feed-forward block: norm, quantize, gate and up, GELU, quantize,
            down, norm, residual add, one entry point each

Everything runs in the library's default summation order, which fixes every
rounding, so the tolerance is "exact" for all kinds.
"""

from __future__ import annotations

import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

HIDDEN, VOCAB, WINDOW, BATCH, PLE, LAYERS = 1536, 262144, 512, 512, 256, 35
EPS = 1e-6
# (N, K) of every product of a token step: the attention projections, the
# feed-forward, the per-layer embedding, the head
SHAPES = ((2048, 1536), (4096, 1536), (256, 1536), (512, 1536), (1536, 2048), (1536, 4096),
          (6144, 1536), (12288, 1536), (1536, 6144), (1536, 12288), (1536, 256), (8960, 1536),
          (262144, 1536))
MODEL_SEED = 20261201

_model_ready = False
_gelu = None


def _pkg():
    """The package (its directory name is not an identifier), from the working folder."""
    if "gemma4_c_amd" not in sys.modules:
        where = os.path.join(os.getcwd(), "gemma4.c_amd")
        spec = importlib.util.spec_from_file_location("gemma4_c_amd", os.path.join(where, "__init__.py"),
                                                      submodule_search_locations=[where])
        module = importlib.util.module_from_spec(spec)
        sys.modules["gemma4_c_amd"] = module
        spec.loader.exec_module(module)
    return sys.modules["gemma4_c_amd"]


def listed():
    return [
        # a short question and the first tokens of its answer: what an interactive user does most
        {"name": "short_turn", "kind": "generate", "prompt": 37, "steps": 16},
        # a long document read in 512-token chunks, then the answer's first tokens (the largest)
        {"name": "document_turn", "kind": "generate", "prompt": 8192, "steps": 8},
        # the head of every decoded token
        {"name": "head_1", "kind": "matmul", "rows": 1, "n": 262144, "k": 1536},
        # a handful of tokens at once (a reply's draft checked, a very short prompt)
        {"name": "down_5", "kind": "matmul", "rows": 5, "n": 1536, "k": 12288},
        # a short prompt's feed-forward product
        {"name": "gate_37", "kind": "matmul", "rows": 37, "n": 12288, "k": 1536},
        # a full chunk's products, both directions of the feed-forward
        {"name": "gate_512", "kind": "matmul", "rows": 512, "n": 6144, "k": 1536},
        {"name": "down_512", "kind": "matmul", "rows": 512, "n": 1536, "k": 12288},
        # one token over a long context, global layer
        {"name": "attend_1_16k", "kind": "attend", "n": 1, "start": 16383, "full": True},
        # a chunk deep inside a long document, global layer
        {"name": "attend_512_8k", "kind": "attend", "n": 512, "start": 7680, "full": True},
        # the attention block of a decoded token (the smallest), and of a ragged
        # turn in a running conversation, window layers past the ring's wrap
        {"name": "layer_1", "kind": "layer", "n": 1, "start": 1500, "full": False},
        {"name": "layer_100", "kind": "layer", "n": 100, "start": 1000, "full": False},
        # the feed-forward block of a short prompt
        {"name": "ffn_64", "kind": "ffn", "rows": 64, "ffn": 6144},
    ]


def _spread(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high + 0.49)))))))


def draw(rng):
    kind = rng.choice(("generate", "matmul", "matmul", "matmul", "attend", "attend", "layer", "layer", "ffn"))
    if kind == "generate":
        return {"kind": kind, "prompt": _spread(rng, 2, 6000), "steps": rng.randint(1, 24)}
    if kind == "matmul":
        n, k = rng.choice(SHAPES)
        # the head runs on one row a token; its many-row form is a dump's
        return {"kind": kind, "rows": _spread(rng, 1, 16 if n == VOCAB else BATCH), "n": n, "k": k}
    full = rng.random() < 0.5
    n = 1 if rng.random() < 0.3 else _spread(rng, 2, BATCH)
    if kind == "attend":
        return {"kind": kind, "n": n, "start": _spread(rng, 1, 24000) - 1, "full": full}
    if kind == "layer":
        return {"kind": kind, "n": n, "start": _spread(rng, 1, 6000) - 1, "full": full}
    return {"kind": kind, "rows": _spread(rng, 1, BATCH), "ffn": rng.choice((6144, 12288))}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(*shape, device="cuda", generator=g)


def _uniform(g, low, high, *shape):
    return torch.rand(*shape, device="cuda", generator=g) * (high - low) + low


class _Weight:
    """A packed matrix on the GPU and its record: int8 values spread as a
    quantized normal's, fp16 scales of N(0, 0.02) weights' size."""

    def __init__(self, g, n, k):
        self.n, self.k = n, k
        self.data = torch.empty(n * k, dtype=torch.int8, device="cuda")
        for i in range(0, n * k, 1 << 26):  # in pieces: the head has 403 M values
            piece = self.data[i:i + (1 << 26)]
            piece.copy_((torch.randn(piece.numel(), device="cuda", generator=g) * 48).round_().clamp_(-127, 127))
        self.scales = _uniform(g, 3e-4, 6e-4, n * k // 64).half()
        self.record = _pkg().Tensor()
        self.record.data, self.record.scales = self.data.data_ptr(), self.scales.data_ptr()
        self.record.shape[0], self.record.shape[1] = n, k

    def double(self, first=0, rows=None):
        """Rows first .. first + rows (multiples of 16) as float64 [rows x k]."""
        n, k = rows or self.n, self.k
        d = self.data[first * k:(first + n) * k].view(n // 16, k // 64, 16, 16, 4)
        d = d.permute(0, 3, 1, 2, 4).reshape(n, k // 64, 64)
        s = self.scales[first * k // 64:(first + n) * k // 64].view(n // 16, k // 64, 16).permute(0, 2, 1)
        return (d.double() * s.reshape(n, k // 64, 1).double()).view(n, k)


def _vector(values):
    r = _pkg().Tensor()
    r.data, r.scales = values.data_ptr(), None
    r.shape[0] = values.shape[0]
    if values.dim() > 1:
        r.shape[1] = values.shape[1]
    return r


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _gelu_table():
    """The exporter's tanh-GELU table over [-8, 8] (exporter.py:73-75)."""
    global _gelu
    if _gelu is None:
        x = np.linspace(-8.0, 8.0, 4096, dtype=np.float32)
        y = 0.5 * x * (1.0 + np.tanh(0.7978845608 * (x + 0.044715 * x * x * x)))
        _gelu = torch.from_numpy(y.astype(np.float32)).cuda()
    return _gelu


def _rope_tables(positions, full):
    hd, pairs, theta = (512, 64, 1e6) if full else (256, 128, 1e4)
    f = theta ** (-2.0 * torch.arange(pairs, device="cuda", dtype=torch.float64) / hd)
    a = torch.arange(positions, device="cuda", dtype=torch.float64)[:, None] * f[None]
    return a.cos().float().contiguous(), a.sin().float().contiguous()


def _ring(case):
    """Positions of the case's KV ring: a power of two that holds what it reads."""
    need = case["start"] + case["n"] if case["full"] else WINDOW + BATCH
    length = 1024
    while length < need:
        length *= 2
    return length


def _load_model():
    """The synthetic E2B-shaped model, once a process: a program loads one
    model, and every turn of it starts at position 0."""
    global _model_ready
    if not _model_ready:
        pkg = _pkg()
        image = pkg.Image.synthetic(seed=MODEL_SEED)
        pkg.check(pkg.lib().g4_init(image.records, 0))
        _model_ready = True


def prepare(case, seed):
    pkg, kind = _pkg(), case["kind"]
    pkg.lib()
    if kind == "generate":
        _load_model()
        gen = np.random.default_rng(int(seed))
        tokens = gen.integers(0, VOCAB, case["prompt"] + case["steps"]).astype(np.int32)
        return {"case": case, "tokens": tokens, "logits": np.empty((1 + case["steps"], VOCAB), np.float32)}
    g = _gen(seed)
    s = {"case": case, "lib": pkg.lib(), "check": pkg.check}
    if kind == "matmul":
        rows, k = case["rows"], case["k"]
        x = _randn(g, rows, k // 64, 64)
        s["xs"] = (x.abs().amax(-1) / 127).contiguous()
        s["xq"] = (x / s["xs"][..., None]).round().clamp(-127, 127).to(torch.int8).view(rows, k).contiguous()
        s["w"] = _Weight(g, case["n"], k)
        s["out"] = torch.empty(rows, case["n"], device="cuda")
    elif kind == "attend":
        # rows as q_norm / k_norm leave them, scores spread by about 4
        hd = 512 if case["full"] else 256
        s["ring"] = _ring(case)
        s["q"] = _randn(g, case["n"], 8 * hd)
        s["keys"] = _randn(g, s["ring"], hd) * (4 / math.sqrt(hd))
        s["values"] = _randn(g, s["ring"], hd)
        s["out"] = torch.empty(case["n"], 8 * hd, device="cuda")
    elif kind == "layer":
        hd = 512 if case["full"] else 256
        s["ring"] = _ring(case)
        s["x"] = _randn(g, case["n"], HIDDEN) * 3
        s["norm"] = _uniform(g, 0.75, 1.25, HIDDEN)
        s["q_norm"] = _uniform(g, 0.75, 1.25, hd)
        s["k_norm"] = _uniform(g, 0.75, 1.25, hd) * (4 / math.sqrt(hd))
        s["w"] = {f: _Weight(g, n, k) for f, n, k in ((10, 8 * hd, HIDDEN), (11, hd, HIDDEN), (12, hd, HIDDEN),
                                                      (13, HIDDEN, 8 * hd))}
        s["cos"], s["sin"] = _rope_tables(case["start"] + case["n"], case["full"])
        s["cache"] = _randn(g, 2, s["ring"], hd)
        s["cache"][0] *= 4 / math.sqrt(hd)
        s["records"] = (pkg.Tensor * 19)()
        s["records"][8], s["records"][9] = _vector(s["q_norm"]), _vector(s["k_norm"])
        for f, w in s["w"].items():
            s["records"][f] = w.record
        s["records"][17], s["records"][18] = _vector(s["cos"]), _vector(s["sin"])
        s["hidden"] = torch.empty_like(s["x"])
    else:
        rows, ffn = case["rows"], case["ffn"]
        s["x"] = _randn(g, rows, HIDDEN) * 3
        s["pre"], s["post"] = _uniform(g, 0.75, 1.25, HIDDEN), _uniform(g, 0.75, 1.25, HIDDEN)
        s["gate"], s["up"], s["down"] = _Weight(g, ffn, HIDDEN), _Weight(g, ffn, HIDDEN), _Weight(g, HIDDEN, ffn)
        s["gelu"] = _gelu_table()
        s["hidden"] = torch.empty(rows, HIDDEN, device="cuda")
        s["a"], s["b"] = torch.empty(rows, ffn, device="cuda"), torch.empty(rows, ffn, device="cuda")
        s["q8"] = torch.empty(rows, ffn, dtype=torch.int8, device="cuda")
        s["qs"] = torch.empty(rows, ffn // 64, device="cuda")
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "generate":
        pkg, lib = _pkg(), _pkg().lib()
        tokens, logits, prompt = s["tokens"], s["logits"], case["prompt"]
        for at in range(0, prompt, BATCH):
            n = min(BATCH, prompt - at)
            pkg.check(lib.g4_forward(tokens[at:].ctypes.data, n, at))
        pkg.check(lib.g4_logits((prompt - 1) % BATCH, logits.ctypes.data))
        for i in range(case["steps"]):
            pkg.check(lib.g4_forward(tokens[prompt + i:].ctypes.data, 1, prompt + i))
            pkg.check(lib.g4_logits(0, logits[1 + i:].ctypes.data))
        return logits
    lib, check, stream = s["lib"], s["check"], _stream()
    if kind == "matmul":
        check(lib.g4_matmul_int8(stream, s["out"].data_ptr(), s["xq"].data_ptr(), s["xs"].data_ptr(),
                                 ctypes.byref(s["w"].record), case["rows"]))
        return s["out"]
    if kind == "attend":
        hd = 512 if case["full"] else 256
        check(lib.g4_attend(stream, s["out"].data_ptr(), s["q"].data_ptr(), s["keys"].data_ptr(),
                            s["values"].data_ptr(), s["ring"], hd, 8, int(case["full"]), case["start"], case["n"]))
        return s["out"]
    if kind == "layer":
        h = s["hidden"].data_ptr()
        check(lib.g4_rmsnorm(stream, h, s["x"].data_ptr(), s["norm"].data_ptr(), HIDDEN, EPS, case["n"]))
        check(lib.g4_attention_layer(stream, h, case["n"], case["start"], s["records"], s["cache"].data_ptr(),
                                     s["ring"], int(case["full"])))
        return s["hidden"], s["cache"]
    rows, ffn, h = case["rows"], case["ffn"], s["hidden"].data_ptr()
    a, b, q8, qs = s["a"].data_ptr(), s["b"].data_ptr(), s["q8"].data_ptr(), s["qs"].data_ptr()
    check(lib.g4_rmsnorm(stream, h, s["x"].data_ptr(), s["pre"].data_ptr(), HIDDEN, EPS, rows))
    check(lib.g4_quantize(stream, q8, qs, h, rows, HIDDEN))
    check(lib.g4_matmul_int8(stream, a, q8, qs, ctypes.byref(s["gate"].record), rows))
    check(lib.g4_matmul_int8(stream, b, q8, qs, ctypes.byref(s["up"].record), rows))
    check(lib.g4_geglu(stream, a, b, rows, ffn, ffn, s["gelu"].data_ptr(), 4096, -8.0, 8.0))
    check(lib.g4_quantize(stream, q8, qs, a, rows, ffn))
    check(lib.g4_matmul_int8(stream, h, q8, qs, ctypes.byref(s["down"].record), rows))
    check(lib.g4_rmsnorm(stream, h, h, s["post"].data_ptr(), HIDDEN, EPS, rows))
    check(lib.g4_add_and_scale(stream, h, s["x"].data_ptr(), rows * HIDDEN, 1.0))
    return s["hidden"]


def _product(rows, n, k):
    """(bytes, operations) of a W8A8 product of quantized rows."""
    return n * k + n * k // 32 + rows * (k + k // 16) + 4 * rows * n, 2 * rows * n * k


def _visible(start, n, full):
    """(sum over the n tokens of the keys they see, distinct keys)."""
    pairs = sum(p + 1 if full else min(p + 1, WINDOW) for p in range(start, start + n))
    return pairs, start + n if full else n + min(start, WINDOW - 1)


def _attention(start, n, full, hd):
    pairs, keys = _visible(start, n, full)
    return 8 * keys * hd + 2 * 4 * n * 8 * hd, 4 * 8 * hd * pairs


def _layer(n, start, full, owner=True):
    hd = 512 if full else 256
    parts = [_product(n, (10 if owner else 8) * hd, HIDDEN), _attention(start, n, full, hd),
             _product(n, HIDDEN, 8 * hd)]
    return sum(p[0] for p in parts), sum(p[1] for p in parts)


def _ffn(rows, ffn):
    parts = [_product(rows, 2 * ffn, HIDDEN), _product(rows, HIDDEN, ffn)]
    return sum(p[0] for p in parts), sum(p[1] for p in parts)


def _pass(start, n):
    """One forward pass: weights once, the activations between layers."""
    total = [_product(n, LAYERS * PLE, HIDDEN)]
    for l in range(LAYERS):
        total += [_layer(n, start, l % 5 == 4, l < 15), _ffn(n, 6144 if l < 15 else 12288),
                  _product(n, PLE, HIDDEN), _product(n, HIDDEN, PLE)]
    return sum(p[0] for p in total), sum(p[1] for p in total)


def work(case):
    kind = case["kind"]
    if kind == "matmul":
        b, f = _product(case["rows"], case["n"], case["k"])
    elif kind == "attend":
        b, f = _attention(case["start"], case["n"], case["full"], 512 if case["full"] else 256)
    elif kind == "layer":
        b, f = _layer(case["n"], case["start"], case["full"])
    elif kind == "ffn":
        b, f = _ffn(case["rows"], case["ffn"])
    else:
        passes = [(at, min(BATCH, case["prompt"] - at)) for at in range(0, case["prompt"], BATCH)]
        passes += [(case["prompt"] + i, 1) for i in range(case["steps"])]
        parts = [_pass(*p) for p in passes] + [_product(1, VOCAB, HIDDEN)] * (1 + case["steps"])
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # The library's default order states every rounding (the order of the sums,
    # fused or separate multiply-adds, libm's own results): another correct
    # implementation gives the same bits.
    return "exact"


def _quantized(x):
    """x after the per-64-value int8 quantization, in the type of x."""
    v = x.view(*x.shape[:-1], x.shape[-1] // 64, 64)
    scale = v.abs().amax(-1, keepdim=True) / 127
    return (torch.where(scale > 0, (v / scale).round(), torch.zeros_like(v)) * scale).view(x.shape)


def _norm(x, w=None):
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
    return y if w is None else y * w.double()


def _attend64(q, keys, values, start, full):
    """q [n x 8 x hd]; keys and values the rings [length x hd]."""
    n, length = q.shape[0], keys.shape[0]
    first = 0 if full else max(0, start - WINDOW + 1)
    at = torch.arange(first, start + n, device="cuda")
    k, v = keys.double()[at & (length - 1)], values.double()[at & (length - 1)]
    out = torch.empty_like(q)
    for t in range(0, n, 64):  # in pieces of 64 tokens
        pos = torch.arange(start + t, start + min(t + 64, n), device="cuda")
        hidden = at[None] > pos[:, None]
        if not full:
            hidden |= at[None] <= pos[:, None] - WINDOW
        piece = q[t:t + 64]
        scores = (piece.reshape(-1, q.shape[-1]) @ k.t()).view(len(pos), 8, -1)
        p = scores.masked_fill(hidden[:, None], -math.inf).softmax(-1)
        out[t:t + 64] = (p.reshape(len(pos) * 8, -1) @ v).view(len(pos), 8, -1)
    return out


def _rotate(x, cos, sin, start):
    """x [n x heads x hd], the half-split rotation of the first pairs."""
    n, pairs, half = x.shape[0], cos.shape[1], x.shape[-1] // 2
    c, s = cos[start:start + n].double()[:, None], sin[start:start + n].double()[:, None]
    y = x.clone()
    a, b = x[..., :pairs], x[..., half:half + pairs]
    y[..., :pairs] = a * c - b * s
    y[..., half:half + pairs] = b * c + a * s
    return y


def exact(case, seed):
    kind = case["kind"]
    if kind == "generate":  # int8 requantizations through 35 layers: no 64-bit value to compare with
        return None
    s = prepare(case, seed)
    if kind == "matmul":
        rows, k = case["rows"], case["k"]
        x = (s["xq"].view(rows, k // 64, 64).double() * s["xs"].double()[..., None]).view(rows, k)
        piece = 16384
        return torch.cat([x @ s["w"].double(i, min(piece, case["n"] - i)).t() for i in range(0, case["n"], piece)], 1)
    if kind == "attend":
        q = s["q"].double().view(case["n"], 8, -1)
        return _attend64(q, s["keys"], s["values"], case["start"], case["full"]).view(case["n"], -1)
    if kind == "layer":
        n, start, full = case["n"], case["start"], case["full"]
        x = _quantized(_norm(s["x"].double(), s["norm"]))
        q = _norm((x @ s["w"][10].double().t()).view(n, 8, -1), s["q_norm"])
        k = _norm((x @ s["w"][11].double().t()).view(n, 1, -1), s["k_norm"])
        v = _norm(x @ s["w"][12].double().t())
        cache = s["cache"].double()
        at = torch.arange(start, start + n, device="cuda") & (s["ring"] - 1)
        cache[0, at] = _rotate(k, s["cos"], s["sin"], start)[:, 0]
        cache[1, at] = v
        out = _attend64(_rotate(q, s["cos"], s["sin"], start), cache[0], cache[1], start, full)
        return _quantized(out.reshape(n, -1)) @ s["w"][13].double().t(), cache
    x = s["x"].double()
    h = _quantized(_norm(x, s["pre"]))
    a, b = h @ s["gate"].double().t(), h @ s["up"].double().t()
    table = s["gelu"].double()
    at = ((a.clamp(-8, 8) + 8) * (4095 / 16)).clamp(max=4094.999999)
    i = at.long()
    act = torch.where(a >= 8, a, table[i] + (at - i) * (table[i + 1] - table[i]))
    return x + _norm(_quantized(act * b) @ s["down"].double().t(), s["post"])
