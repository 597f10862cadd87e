"""Performance cases of the W4A4 layers: the work a program does with this package.

Every case goes through the package's public entry points with weights in the form that the
loader (``apply.load_time_weight``) keeps them, as ``apply_w4a4_from_dir`` leaves a model:

* ``linear``    one ``W4A4Linear`` (any K that is a multiple of 64, MFMA-layout or row-major
                reference-layout weights): the projections of a model that is not fused;
* ``qkv``       input RMSNorm + the three QKV projections with one shared activation quant;
* ``gate_up``   post-attention RMSNorm + gate/up with the GELU-tanh * up epilogue;
* ``down``      the K = 16384 down projection with the residual add;
* ``attention`` RoPE + grouped-query attention of a prefix (8 query heads, 1 KV head of 256);
* ``layer``     a whole PaliGemma-2B-shaped decoder layer, called eagerly, or replayed as
                the captured graph that a latency-bound server keeps (``replay``: the new
                hidden states are copied into the graph's input on every pass).

Rows are batch * tokens.  Sizes are PaliGemma-2B's prefix LM (hidden 2048, intermediate
16384, 776-token prefixes, batch 1 to 8) and the widths of this repository's tests.
Activations are N(0, 1) with 1% of the channels 20 times larger, the down projection's are
gelu_tanh(N(0, 1)) * N(0, 1), and the weights have the code statistics of a packed N(0, 0.02)
weight.  The decoder layer's hidden states are 8 times larger, as residual streams are a few
layers in (its updates are then a fraction of the stream).

Arithmetic.  The activation codes are decided by a rounding to 4 bits, so a difference in the
last bit of a layer's input can move a code by one; ``exact`` therefore rounds to fp16
where the layer's tensors are fp16 (the norm's output, the GELU's, q/k/v, the attention's)
and computes everything between in 64 bits.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "pi05-pytorch-fast_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

HIDDEN, INTER, HEADS, HEAD_DIM = 2048, 16384, 8, 256
ROTATED = (1024, 2048, 16384)
EPS = 1e-6


def listed():
    return [
        # a single token through one projection: the latency of a call
        {"name": "linear_1row", "op": "linear", "rows": 1, "k": 2048, "n": 2048, "layout": "mfma"},
        # another model's width (no rotation) on weights as the reference stores them
        {"name": "linear_1000x4096", "op": "linear", "rows": 1000, "k": 4096, "n": 1024, "layout": "row"},
        # a short prompt's QKV
        {"name": "qkv_64", "op": "qkv", "rows": 64},
        # one camera's tokens and a short prompt through the MLP's first half
        {"name": "gate_up_200", "op": "gate_up", "rows": 200},
        # the 776-token prefix (three cameras and a prompt): the headline's largest GEMM
        {"name": "gate_up_776", "op": "gate_up", "rows": 776},
        # the same prefix's down projection
        {"name": "down_776", "op": "down", "rows": 776},
        # ragged prefixes of a few requests, with padding keys
        {"name": "attention_3x389", "op": "attention", "batch": 3, "tokens": 389, "mask": True},
        # a batch of full prefixes
        {"name": "attention_8x776", "op": "attention", "batch": 8, "tokens": 776, "mask": True},
        # a decoder layer of the headline forward, as it is served
        {"name": "layer_776", "op": "layer", "batch": 1, "tokens": 776, "mask": False, "replay": True},
        # the throughput point: batch 8 x 776 tokens, its two MLP halves and the whole layer
        {"name": "gate_up_8x776", "op": "gate_up", "rows": 6208},
        {"name": "down_8x776", "op": "down", "rows": 6208},
        {"name": "layer_8x776", "op": "layer", "batch": 8, "tokens": 776, "mask": True, "replay": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["linear", "linear", "qkv", "gate_up", "gate_up", "down", "down", "attention", "layer", "layer"])
    if op == "linear":
        return {"op": op, "rows": _log(rng, 1, 6208), "k": rng.choice([512, 1024, 2048, 4096, 192]),
                "n": 16 * _log(rng, 4, 256), "layout": rng.choice(["mfma", "row"])}
    if op in ("qkv", "gate_up", "down"):
        return {"op": op, "rows": _log(rng, 1, 6208)}
    if op == "attention":
        return {"op": op, "batch": rng.randint(1, 8), "tokens": _log(rng, 8, 776), "mask": rng.random() < 0.7}
    batch = rng.randint(1, 8)
    return {"op": op, "batch": batch, "tokens": _log(rng, 32, 776), "mask": rng.random() < 0.5, "replay": batch == 1}


# ------------------------------------------------------------------ inputs, from the seed
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(0x5EED + int(seed))


def _weight(gen, n, k):
    """INT4 codes [N, K] (int8, in [-7, 7]) and fp32 column scales [N]."""
    codes = torch.randn((n, k), device="cuda", generator=gen).mul_(2.0).round_().clamp_(-7, 7).to(torch.int8)
    return codes, (torch.rand((n,), device="cuda", generator=gen) * 0.2 + 0.9) * 0.01


def _pack(codes, scale):
    """The reference's row-major packed form, int32 [N, K/8 + 1]."""
    nib = codes.to(torch.int32).view(codes.size(0), -1, 8) & 0xF
    word = torch.zeros(nib.shape[:2], dtype=torch.int32, device="cuda")
    for j in range(8):
        word |= nib[..., j] << (4 * j)
    return torch.cat([word, scale.view(torch.int32)[:, None]], dim=1)


def _activations(gen, *shape):
    x = torch.randn(shape, device="cuda", generator=gen)
    cols = torch.randperm(shape[-1], device="cuda", generator=gen)[: max(1, shape[-1] // 100)]
    x[..., cols] *= 20.0
    return x


def _norm_weight(gen):
    return (torch.randn((HIDDEN,), device="cuda", generator=gen) * 0.05).half()


def _rotary(batch, tokens):
    inv = 1.0 / (10000.0 ** (torch.arange(0, HEAD_DIM, 2, device="cuda").float() / HEAD_DIM))
    ang = torch.arange(tokens, device="cuda").float()[:, None] * inv[None]
    emb = torch.cat([ang, ang], dim=-1)[None].expand(batch, tokens, HEAD_DIM)
    return emb.cos().half().contiguous(), emb.sin().half().contiguous()


def _mask(gen, batch, tokens):
    """Additive fp16 mask [B, 1, S, S] of a bidirectional prefix: padding keys at the end of
    each sequence (at most a quarter of it) are masked for every query."""
    keep = torch.randint(max(1, tokens - tokens // 4), tokens + 1, (batch,), device="cuda", generator=gen)
    pad = torch.arange(tokens, device="cuda")[None] >= keep[:, None]
    row = torch.zeros((batch, tokens), dtype=torch.float16, device="cuda").masked_fill_(pad, torch.finfo(torch.float16).min)
    return row[:, None, None, :].expand(batch, 1, tokens, tokens).contiguous()


_LAYER = (("self_attn.q_proj", HIDDEN, HIDDEN), ("self_attn.k_proj", HEAD_DIM, HIDDEN), ("self_attn.v_proj", HEAD_DIM, HIDDEN),
          ("self_attn.o_proj", HIDDEN, HIDDEN), ("mlp.gate_proj", INTER, HIDDEN), ("mlp.up_proj", INTER, HIDDEN),
          ("mlp.down_proj", HIDDEN, INTER))


def _inputs(case, seed):
    """Everything a case is made of: weights as (codes, scales), activations and tables."""
    gen, op = _gen(seed), case["op"]
    s = {}
    if op == "linear":
        s["w"] = _weight(gen, case["n"], case["k"])
        s["x"] = _activations(gen, case["rows"], case["k"]).half()
    elif op == "qkv":
        s["ws"] = [_weight(gen, n, HIDDEN) for n in (HIDDEN, HEAD_DIM, HEAD_DIM)]
        s["norm"] = _norm_weight(gen)
        s["x"] = _activations(gen, case["rows"], HIDDEN).half()
    elif op == "gate_up":
        s["ws"] = [_weight(gen, INTER, HIDDEN) for _ in range(2)]
        s["norm"] = _norm_weight(gen)
        s["x"] = _activations(gen, case["rows"], HIDDEN).half()
    elif op == "down":
        s["w"] = _weight(gen, HIDDEN, INTER)
        g = torch.randn((case["rows"], INTER), device="cuda", generator=gen)
        u = torch.randn((case["rows"], INTER), device="cuda", generator=gen)
        s["x"] = (torch.nn.functional.gelu(g, approximate="tanh") * u).half()
        s["res"] = _activations(gen, case["rows"], HIDDEN).half()
    else:
        b, t = case["batch"], case["tokens"]
        s["cos"], s["sin"] = _rotary(b, t)
        s["mask"] = _mask(gen, b, t) if case["mask"] else None
        if op == "attention":
            s["q"] = torch.randn((b, t, HEADS * HEAD_DIM), device="cuda", generator=gen).half()
            s["k"] = torch.randn((b, t, HEAD_DIM), device="cuda", generator=gen).half()
            s["v"] = torch.randn((b, t, HEAD_DIM), device="cuda", generator=gen).half()
        else:
            s["ws"] = {name: _weight(gen, n, k) for name, n, k in _LAYER}
            s["norm"], s["norm2"] = _norm_weight(gen), _norm_weight(gen)
            s["x"] = (_activations(gen, b, t, HIDDEN) * 8.0).half()
    return s


# ------------------------------------------------------------------ the calls
@torch.no_grad()
def prepare(case, seed):
    from pi05_fast.w4a4 import W4A4Linear, extension
    from pi05_fast.w4a4.apply import load_time_weight

    extension.preload()
    s, op = _inputs(case, seed), case["op"]
    s["op"] = op
    dev = torch.device("cuda")

    def load(w, name):
        codes, scale = w
        return load_time_weight(_pack(codes, scale), name, codes.size(1), codes.size(0), dev)[0]

    if op == "linear":
        codes, scale = s.pop("w")
        w = _pack(codes, scale) if case["layout"] == "row" else load((codes, scale), "layers.0.self_attn.o_proj")
        s["module"] = W4A4Linear(w, in_features=case["k"])
    elif op == "qkv":
        s["ws"] = [load(w, f"layers.0.self_attn.{p}_proj") for w, p in zip(s["ws"], "qkv")]
    elif op == "gate_up":
        s["ws"] = [load(w, f"layers.0.mlp.{p}_proj") for w, p in zip(s["ws"], ("gate", "up"))]
    elif op == "down":
        s["w"] = load(s["w"], "layers.0.mlp.down_proj")
    elif op == "layer":
        from pi05_fast.w4a4.prefix_lm import build_prefix_lm

        packed = {f"layers.0.{name}": _pack(*w) for name, w in s.pop("ws").items()}
        model, _ = build_prefix_lm(dev, num_layers=1, packed=packed)
        layer = model.layers[0]
        layer.input_layernorm.weight.copy_(s["norm"])
        layer.post_attention_layernorm.weight.copy_(s["norm2"])
        s["layer"] = layer
        if case["replay"]:
            static = s["x"].clone()
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                for _ in range(2):
                    _layer(s, static)
            torch.cuda.current_stream().wait_stream(side)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                out = _layer(s, static)
            s["static"], s["graph"], s["out"] = static, graph, out
    return s


def _layer(s, x):
    return s["layer"](x, attention_mask=s["mask"], position_embeddings=(s["cos"], s["sin"]))


@torch.no_grad()
def run(s):
    from pi05_fast.w4a4 import extension as ext

    op = s["op"]
    if op == "linear":
        return s["module"](s["x"])
    if op == "qkv":
        return ext.rms_norm_int4_gemm3(s["x"], s["norm"], EPS, *s["ws"])
    if op == "gate_up":
        return ext.rms_norm_int4_gemm2_gelu(s["x"], s["norm"], EPS, *s["ws"])
    if op == "down":
        return ext.int4_gemm_residual(s["x"], s["w"], s["res"])
    if op == "attention":
        return ext.prefix_attention(s["q"], s["k"], s["v"], s["cos"], s["sin"], s["mask"], HEAD_DIM**-0.5, HEADS, 1)
    if "graph" in s:
        s["static"].copy_(s["x"])
        s["graph"].replay()
        return s["out"]
    return _layer(s, s["x"])


# ------------------------------------------------------------------ what a pass cannot do without
def _gemm_work(rows, k, n):
    return {"bytes": n * k / 2 + 4 * n, "flops": 2.0 * rows * k * n}


def _attention_work(b, t, mask):
    # q in, out out, k/v in, key states out, rotary tables, mask
    return {"bytes": 2.0 * b * t * (2 * HEADS * HEAD_DIM + 5 * HEAD_DIM + (t if mask else 0)),
            "flops": 4.0 * b * HEADS * t * t * HEAD_DIM}


def work(case):
    op = case["op"]
    if op == "linear":
        m, k, n = case["rows"], case["k"], case["n"]
        w = _gemm_work(m, k, n)
        return {"bytes": w["bytes"] + 2.0 * m * (k + n), "flops": w["flops"]}
    if op in ("qkv", "gate_up", "down"):
        m = case["rows"]
        k, n, cols = {"qkv": (HIDDEN, HIDDEN + 2 * HEAD_DIM, HIDDEN + 2 * HEAD_DIM),
                      "gate_up": (HIDDEN, 2 * INTER, INTER), "down": (INTER, HIDDEN, 2 * HIDDEN)}[op]
        w = _gemm_work(m, k, n)
        return {"bytes": w["bytes"] + 2.0 * m * (k + cols), "flops": w["flops"]}
    b, t = case["batch"], case["tokens"]
    att = _attention_work(b, t, case["mask"])
    if op == "attention":
        return att
    gemms = [_gemm_work(b * t, k, n) for _, n, k in _LAYER]
    rows = 2.0 * b * t * (2 * HIDDEN + 2 * HEAD_DIM + (t if case["mask"] else 0))  # hidden in and out, tables, mask
    return {"bytes": rows + sum(g["bytes"] for g in gemms), "flops": att["flops"] + sum(g["flops"] for g in gemms)}


def tolerance(case):
    """About four times the distance from ``exact`` that was measured.  Products of codes: an
    fp16 output ulp (2.1e-4 in the 2-norm), and a code that moves by one here and there after a
    transform in another order (behind the norm: up to 7e-4, behind the GELU too: up to
    2.3e-3).  Without a
    rotation, values of a few significant bits often lie exactly between two codes, and the last
    bit of the row's scale decides (6.1e-3).  The attention adds the fp16 rounding of its
    probabilities (5.4e-4).  The decoder layer quantizes to 4 bits after its attention and
    again after the GELU, so another rounding of the attention's output moves codes of
    every later stage (4.5e-3)."""
    op = case["op"]
    if op == "layer":
        return {"rel": 1.8e-2, "max": 0.2}
    if op == "attention":
        return {"rel": 2.2e-3, "max": 0.03}
    if op == "linear" and case["k"] not in ROTATED:
        return {"rel": 2.4e-2, "max": 0.5}
    if op == "gate_up":
        return {"rel": 9e-3, "max": 0.3}
    if op == "qkv":
        return {"rel": 3e-3, "max": 0.2}
    return {"rel": 1e-3, "max": 0.1}


# ------------------------------------------------------------------ 64-bit results
def _r16(x):
    return x.half().double()


def _fwht(x):
    n, h = x.size(-1), 1
    while h < n:
        y = x.view(-1, n // (2 * h), 2, h)
        x = torch.stack((y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]), dim=2).view(-1, n)
        h *= 2
    return x


def _quant(x):
    """Codes and row scales of [M, K] rows (64 bits)."""
    k = x.size(-1)
    root = 1.0
    if k in ROTATED:
        x, root = _fwht(x), 1.0 / math.sqrt(k)
    step = x.abs().amax(dim=-1, keepdim=True) / 7.0 + 1e-12
    return torch.round(x / step).clamp_(-7, 7), step * root


def _product(q, w):
    codes, scale = w
    a, sa = q
    return (a @ codes.double().t().contiguous()) * sa * scale.double()[None]


def _rms(x, weight):
    return _r16(x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * (1.0 + weight.double()))


def _gelu_up(q, w_gate, w_up):
    gate = _r16(_product(q, w_gate))
    return _r16(torch.nn.functional.gelu(gate, approximate="tanh")) * _r16(_product(q, w_up))


def _rope(x, cos, sin):
    """x [B, S, H, 256] with tables [B, S, 256]."""
    half = x.size(-1) // 2
    rot = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return _r16(_r16(x * cos[:, :, None]) + _r16(rot * sin[:, :, None]))


def _attend(q, k, v, cos, sin, mask):
    """(output [B, S, H * 256], key states [B, 1, S, 256]) with one KV head."""
    b, t, _ = q.shape
    cos, sin = cos.double(), sin.double()
    q = _rope(q.view(b, t, HEADS, HEAD_DIM), cos, sin)
    k = _rope(k.view(b, t, 1, HEAD_DIM), cos, sin)
    out = torch.empty_like(q)
    for i in range(b):
        kt = k[i, :, 0].t().contiguous()
        for h in range(HEADS):
            score = (q[i, :, h].contiguous() @ kt) * HEAD_DIM**-0.5
            if mask is not None:
                score = score + mask[i, 0].double()
            out[i, :, h] = torch.softmax(score, dim=-1) @ v[i].contiguous()
    return out.view(b, t, HEADS * HEAD_DIM), k.transpose(1, 2).contiguous()


@torch.no_grad()
def exact(case, seed):
    s, op = _inputs(case, seed), case["op"]
    if op == "linear":
        return _product(_quant(s["x"].double()), s["w"])
    if op == "qkv":
        q = _quant(_rms(s["x"].double(), s["norm"]))
        return tuple(_product(q, w) for w in s["ws"])
    if op == "gate_up":
        return _gelu_up(_quant(_rms(s["x"].double(), s["norm"])), *s["ws"])
    if op == "down":
        return _r16(_product(_quant(s["x"].double()), s["w"])) + s["res"].double()
    if op == "attention":
        return _attend(s["q"].double(), s["k"].double(), s["v"].double(), s["cos"], s["sin"], s["mask"])
    b, t = case["batch"], case["tokens"]
    x = s["x"].double().view(b * t, HIDDEN)
    w = s["ws"]
    qa = _quant(_rms(x, s["norm"]))
    q, k, v = (_r16(_product(qa, w[f"self_attn.{p}_proj"])).view(b, t, -1) for p in "qkv")
    att = _r16(_attend(q, k, v, s["cos"], s["sin"], s["mask"])[0]).view(b * t, HIDDEN)
    x = _r16(_r16(_product(_quant(att), w["self_attn.o_proj"])) + x)
    h = _r16(_gelu_up(_quant(_rms(x, s["norm2"])), w["mlp.gate_proj"], w["mlp.up_proj"]))
    return (_r16(_product(_quant(h), w["mlp.down_proj"])) + x).view(b, t, HIDDEN)
