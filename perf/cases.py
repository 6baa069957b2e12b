"""Timing cases of the attention path and its projections, over the ranges a serving program meets.

Five kinds of case, each through the package's public entry points:

  decode   one token of 1..16 sequences through a full-attention layer (KVCache.full_core): the step of a decode loop
  prefill  a prompt, or a piece of one after a cached prefix, through a full-attention layer (KVCache.attn_prefill)
  linear   linear_core of a Gated-DeltaNet layer: one token of a batch of sequences, or a prompt of one sequence
  proj     a layer's weight projections for a number of tokens (Context.quantize_project_q8_k, or gemv_f32 for the types
           that a file keeps at higher precision), every input independent of the other projections' outputs
  token    the layer cores of a whole token, recorded once as a graph and replayed at the token's position (DecodeGraph)
"""
import importlib.util
import math
import os
import re
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "qwen3.8_27b_in_rust_amd")

HEADS, KV_HEADS, HEAD_DIM, KV_DIM, Q_DIM, QG_DIM = 24, 4, 256, 1024, 6144, 12288
LIN_QK, LIN_V, LIN_DIM, QKV_DIM = 16, 48, 128, 10240
STATE, CONV = LIN_V * LIN_DIM * LIN_DIM, QKV_DIM * 3
PAGE = 16
HIDDEN, FFN = 5120, 17408

# ggml type: bytes of a block, weights of a block, offsets of its f16 scales
BLOCKS = {10: (84, 256, (80, 82)), 11: (110, 256, (108,)), 12: (144, 256, (0, 2)), 13: (176, 256, (0, 2)),
          14: (210, 256, (208,)), 21: (110, 256, (0,)), 22: (82, 256, (0,)), 23: (136, 256, (0,)), 8: (34, 32, (0,))}
BF16, F32, Q8_0 = 30, 0, 8
# what a model file of each mix holds: the type of its matrices and that of the down projection, kept finer
MIXES = {"q4_k_m": (12, 14), "q5_k_m": (13, 14), "q3_k_m": (11, 12), "q2_k": (10, 11), "iq4_xs": (23, 13),
         "iq2_m": (22, 21), "q8_0": (Q8_0, Q8_0), "bf16": (BF16, BF16)}
IQ4 = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)


def listed():
    return [
        # a chat's decode step early in its context: two short launches, latency counts
        {"name": "decode_1k", "kind": "decode", "seqs": 1, "ctx": 1021},
        # the decode step of a long document, batch 1
        {"name": "decode_32k", "kind": "decode", "seqs": 1, "ctx": 32768},
        # a server's step: 16 sequences of ragged lengths, the longest 32K
        {"name": "decode_batch16", "kind": "decode", "seqs": 16, "ctx": 32768},
        # a whole prompt at once
        {"name": "prefill_4096", "kind": "prefill", "base": 0, "tokens": 4096},
        # the next piece of a prompt that is fed in pieces, a ragged size
        {"name": "prefill_509_after_6000", "kind": "prefill", "base": 6000, "tokens": 509},
        # DeltaNet: a whole prompt, a short ragged one, and a batch's decode step
        {"name": "linear_4096", "kind": "linear", "seqs": 1, "tokens": 4096},
        {"name": "linear_331", "kind": "linear", "seqs": 1, "tokens": 331},
        {"name": "linear_decode_batch8", "kind": "linear", "seqs": 8, "tokens": 1},
        # the projections around a full-attention layer: one token, a few tokens (a small batch, or a draft verified),
        # and the FFN's of a long prompt
        {"name": "proj_1", "kind": "proj", "layer": "full", "tokens": 1, "mix": "q4_k_m"},
        {"name": "proj_6", "kind": "proj", "layer": "full", "tokens": 6, "mix": "q4_k_m"},
        {"name": "proj_ffn_3001", "kind": "proj", "layer": "ffn", "tokens": 3001, "mix": "q4_k_m"},
        # a token of the 64-layer hybrid: 48 DeltaNet and 16 full-attention layers, 4K of context
        {"name": "token_64_layers", "kind": "token", "layers": 64, "seqs": 1, "ctx": 4099},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("decode", "prefill", "linear", "proj", "proj", "token"))
    if kind == "decode":
        return {"kind": kind, "seqs": _log_int(rng, 1, 16), "ctx": _log_int(rng, 64, 32768)}
    if kind == "prefill":
        tokens = _log_int(rng, 16, 4096)
        most = 4096 * 4096 // tokens  # as much work as 4096 tokens after 2048 at the most
        return {"kind": kind, "base": rng.choice((0, _log_int(rng, 16, min(16384, most)))), "tokens": tokens}
    if kind == "linear":
        if rng.random() < 0.4:
            return {"kind": kind, "seqs": _log_int(rng, 1, 32), "tokens": 1}
        return {"kind": kind, "seqs": 1, "tokens": _log_int(rng, 16, 4096)}
    if kind == "proj":
        mix = rng.choice(("q4_k_m", "q4_k_m", "q4_k_m") + tuple(sorted(MIXES)))
        few = rng.random() < 0.6
        layer = rng.choice(("full", "linear", "ffn"))
        most = {"bf16": 1000, "q8_0": 1000}.get(mix, 1700)
        return {"kind": kind, "layer": layer, "tokens": rng.randint(1, 8) if few else _log_int(rng, 9, most), "mix": mix}
    return {"kind": kind, "layers": 4 * rng.randint(1, 16), "seqs": rng.choice((1, 1, 2, 3)),
            "ctx": _log_int(rng, 64, 4096)}


# ------------------------------------------------------------------ the program's side

_held = {}


def _pkg():
    if "q38amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location("q38amd", os.path.join(PKG_DIR, "__init__.py"),
                                                      submodule_search_locations=[PKG_DIR])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["q38amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["q38amd"]


def _ctx():
    """The program's one context."""
    if "ctx" not in _held:
        _held["ctx"] = _pkg().Context(0)
    return _held["ctx"]


class _State:
    """Buffers and handles of one case; the cache and graph are given back with it."""

    def __init__(self, case):
        self.case, self.kv, self.graph = case, None, None

    def __del__(self):
        for h in (self.graph, self.kv):
            if h is not None:
                h.close()


class _Gen:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, sigma=1.0, mean=0.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)
        return x.mul_(sigma).add_(mean) if (sigma, mean) != (1.0, 0.0) else x

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda", dtype=torch.float32).mul_(hi - lo).add_(lo)

    def bytes(self, *shape):
        return torch.randint(0, 256, shape, generator=self.g, device="cuda", dtype=torch.uint8)


def _contexts(case):
    """The sequences' lengths: the longest, then down to a sixteenth of it, evenly over the logarithm."""
    n, ctx = case["seqs"], case["ctx"]
    return [max(17, int(ctx * 16.0 ** (-i / max(1, n - 1)))) - (i & 7) for i in range(n)]


def _attention_inputs(g, n):
    """Raw projections of one token of n sequences, and the layer's norm weights."""
    return {"q_norm": g.normal(HEAD_DIM, sigma=0.1, mean=1.0), "k_norm": g.normal(HEAD_DIM, sigma=0.1, mean=1.0),
            "qg": g.normal(n, QG_DIM), "key": g.normal(n, KV_DIM), "value": g.normal(n, KV_DIM)}


def _linear_inputs(g, seqs, tokens):
    """A DeltaNet layer's weights, states and raw projections."""
    n = seqs * tokens
    return {"conv_w": g.normal(QKV_DIM, 4, sigma=0.3), "dt": g.normal(LIN_V, sigma=0.1),
            "a": g.uniform(-1.0, -0.02, LIN_V), "norm": g.normal(LIN_DIM, sigma=0.1, mean=1.0),
            "conv": g.normal(seqs, QKV_DIM, 3), "delta": g.normal(seqs, LIN_V, LIN_DIM, LIN_DIM, sigma=0.02),
            "qkv": g.normal(n, QKV_DIM), "z": g.normal(n, Q_DIM), "beta": g.normal(n, LIN_V), "alpha": g.normal(n, LIN_V)}


def _groups(case):
    """The projections of a layer: (ggml type, rows of each matrix of one input, width)."""
    ty, fine = MIXES[case["mix"]]
    ffn = [(ty, (FFN, FFN), HIDDEN), (fine, (HIDDEN,), FFN)]
    if case["layer"] == "ffn":
        return ffn
    if case["layer"] == "full":
        return [(ty, (QG_DIM, KV_DIM, KV_DIM), HIDDEN), (ty, (HIDDEN,), Q_DIM)] + ffn
    return [(ty, (QKV_DIM, Q_DIM), HIDDEN), (F32, (LIN_V, LIN_V), HIDDEN), (ty, (HIDDEN,), Q_DIM)] + ffn


def _row_bytes(ty, width):
    return width * 4 if ty == F32 else width * 2 if ty == BF16 else width // BLOCKS[ty][1] * BLOCKS[ty][0]


def _weights(g, ty, rows, width):
    """Random rows of a format, its f16 scales of a trained matrix's size."""
    if ty == F32:
        return g.normal(rows, width, sigma=0.02)
    if ty == BF16:
        return g.normal(rows, width, sigma=0.02).to(torch.bfloat16)
    size, per, at = BLOCKS[ty]
    w = g.bytes(rows * (width // per), size)
    for o in at:
        w[:, o:o + 2] = g.uniform(2e-4, 2e-3, w.shape[0], 1).to(torch.float16).view(torch.uint8)
    return w


def _fill(kv, layer, seq, k, v):
    kv.write(layer, seq, 0, k.shape[0], k.data_ptr(), v.data_ptr())


def _new_kv(ctx, n_slots, ctxs):
    pages = [-(-c // PAGE) for c in ctxs]
    return _pkg().KVCache(ctx, n_slots=n_slots, max_pages=sum(pages), max_seqs=len(ctxs),
                          max_tokens_per_seq=max(pages) * PAGE)


def prepare(case, seed):
    ctx, g, s = _ctx(), _Gen(seed), _State(case)
    kind = case["kind"]
    new = lambda *shape: torch.zeros(shape, device="cuda", dtype=torch.float32)  # noqa: E731
    if kind == "decode":
        s.ctxs = _contexts(case)
        s.kv = _new_kv(ctx, 1, s.ctxs)
        s.seqs = [s.kv.seq_create() for _ in s.ctxs]
        s.x = _attention_inputs(g, len(s.ctxs))
        for seq, c in zip(s.seqs, s.ctxs):
            k, v = g.normal(c - 1, KV_DIM), g.normal(c - 1, KV_DIM)
            torch.cuda.synchronize()
            _fill(s.kv, 3, seq, k, v)
            ctx.sync()
        s.out = new(len(s.ctxs), Q_DIM)
    elif kind == "prefill":
        base, n = case["base"], case["tokens"]
        s.kv = _new_kv(ctx, 1, [base + n])
        s.seq = s.kv.seq_create()
        s.x = _prefill_inputs(g, base, n)
        s.out = new(n, Q_DIM)
        # the prefix went through the same layer, piece by piece
        for at in range(0, base, 2048):
            m = min(2048, base - at)
            q, o = g.normal(m, Q_DIM), new(m, Q_DIM)
            torch.cuda.synchronize()
            s.kv.attn_prefill(3, s.seq, at, m, q.data_ptr(), s.x["k"][at:].data_ptr(), s.x["v"][at:].data_ptr(), o.data_ptr())
            ctx.sync()
    elif kind == "linear":
        s.x = _linear_inputs(g, case["seqs"], case["tokens"])
        s.out = new(case["seqs"] * case["tokens"], Q_DIM)
    elif kind == "proj":
        s.groups = []
        for ty, rows, width in _groups(case):
            ws = [_weights(g, ty, r, width) for r in rows]
            x = g.normal(case["tokens"], width)
            outs = [new(case["tokens"], r) for r in rows]
            q = None
            if ty in BLOCKS and BLOCKS[ty][1] == 256:
                q = torch.zeros(ctx.q8k_bytes(case["tokens"], width), device="cuda", dtype=torch.uint8)
            s.groups.append((ty, rows, width, ws, x, q, outs))
    else:
        _prepare_token(ctx, g, s, new)
    torch.cuda.synchronize()
    return s


def _prefill_inputs(g, base, n):
    return {"q": g.normal(n, Q_DIM), "gate": g.normal(n, Q_DIM), "k": g.normal(base + n, KV_DIM), "v": g.normal(base + n, KV_DIM)}


def _prepare_token(ctx, g, s, new):
    case = s.case
    n = case["seqs"]
    s.ctxs = _contexts(case)
    s.kv = _new_kv(ctx, case["layers"] // 4, s.ctxs)
    s.seqs = [s.kv.seq_create() for _ in s.ctxs]
    s.positions = [c - 1 for c in s.ctxs]
    linear = case["layers"] // 4 * 3
    s.x, s.outs = [], new(case["layers"], n, Q_DIM)
    s.conv, s.delta = new(linear, n, QKV_DIM, 3), new(linear, n, LIN_V, LIN_DIM, LIN_DIM)
    at = 0
    for layer in range(case["layers"]):
        if layer % 4 == 3:
            x = _attention_inputs(g, n)
            for seq, c in zip(s.seqs, s.ctxs):
                k, v = g.normal(c - 1, KV_DIM), g.normal(c - 1, KV_DIM)
                torch.cuda.synchronize()
                _fill(s.kv, layer, seq, k, v)
                ctx.sync()
        else:
            x = _linear_inputs(g, n, 1)
            for name, every in (("conv", s.conv), ("delta", s.delta)):
                every[at].copy_(x[name])
                x[name] = every[at]
            at += 1
        s.x.append(x)
    torch.cuda.synchronize()
    s.graph = s.kv.decode_graph(s.seqs, s.positions)
    for layer, x in enumerate(s.x):
        p, out = {k: v.data_ptr() for k, v in x.items()}, s.outs[layer].data_ptr()
        if layer % 4 == 3:
            s.graph.add_decode({"layer": layer, "q": p["qg"], "k_new": p["key"], "v_new": p["value"], "q_norm": p["q_norm"],
                                "k_norm": p["k_norm"], "out": out})
        else:
            s.graph.add_linear_core(n, p["conv_w"], p["dt"], p["a"], p["norm"], p["conv"], p["delta"], p["qkv"], p["z"],
                                    p["beta"], p["alpha"], out)
    s.graph.end()


def run(s):
    ctx, case = _ctx(), s.case
    kind = case["kind"]
    if kind == "decode":
        x = s.x
        s.kv.full_core(3, s.seqs, [c - 1 for c in s.ctxs], x["q_norm"].data_ptr(), x["k_norm"].data_ptr(), x["qg"].data_ptr(),
                       x["key"].data_ptr(), x["value"].data_ptr(), s.out.data_ptr())
        return s.out
    if kind == "prefill":
        x, base = s.x, case["base"]
        s.kv.attn_prefill(3, s.seq, base, case["tokens"], x["q"].data_ptr(), x["k"][base:].data_ptr(), x["v"][base:].data_ptr(),
                          s.out.data_ptr(), gate=x["gate"].data_ptr())
        return s.out
    if kind == "linear":
        x = {k: v.data_ptr() for k, v in s.x.items()}
        ctx.linear_core(case["seqs"], case["tokens"], x["conv_w"], x["dt"], x["a"], x["norm"], x["conv"], x["delta"], x["qkv"],
                        x["z"], x["beta"], x["alpha"], s.out.data_ptr())
        return {"out": s.out, "conv": s.x["conv"], "delta": s.x["delta"]}
    if kind == "proj":
        result = []
        for ty, rows, width, ws, x, q, outs in s.groups:
            if q is None:
                for r, w, o in zip(rows, ws, outs):
                    ctx.gemv_f32(ty, r, width, w.data_ptr(), x.data_ptr(), case["tokens"], o.data_ptr())
                result.append({"outs": outs})
            else:
                ctx.quantize_project_q8_k(ty, rows, width, [w.data_ptr() for w in ws], x.data_ptr(), case["tokens"],
                                          q.data_ptr(), [o.data_ptr() for o in outs])
                result.append({"outs": outs, "q8k": q})
        return result
    s.graph.set_positions(s.positions)
    s.graph.launch()
    return {"outs": s.outs, "conv": s.conv, "delta": s.delta}


# ------------------------------------------------------------------ what a pass cannot do without


def _decode_work(ctxs):
    n = len(ctxs)
    return {"bytes": sum(ctxs) * 2 * KV_DIM * 4 + n * 4 * (QG_DIM + 2 * KV_DIM + Q_DIM), "flops": sum(ctxs) * HEADS * HEAD_DIM * 4}


def _linear_work(seqs, tokens):
    n = seqs * tokens
    weights = 4 * (QKV_DIM * 4 + 2 * LIN_V + LIN_DIM)
    return {"bytes": 8 * seqs * (STATE + CONV) + 4 * n * (QKV_DIM + 2 * Q_DIM + 2 * LIN_V) + weights,
            "flops": n * LIN_V * LIN_DIM * LIN_DIM * 6}


def work(case):
    kind = case["kind"]
    if kind == "decode":
        return _decode_work(_contexts(case))
    if kind == "prefill":
        base, n = case["base"], case["tokens"]
        return {"bytes": 4 * (2 * KV_DIM * (base + 2 * n) + 3 * n * Q_DIM),
                "flops": HEADS * HEAD_DIM * 4 * (n * base + n * (n + 1) // 2)}
    if kind == "linear":
        return _linear_work(case["seqs"], case["tokens"])
    if kind == "proj":
        b = f = 0
        for ty, rows, width in _groups(case):
            b += sum(rows) * _row_bytes(ty, width) + 4 * case["tokens"] * (width + sum(rows))
            f += 2 * case["tokens"] * sum(rows) * width
        return {"bytes": b, "flops": f}
    a, l = _decode_work(_contexts(case)), _linear_work(case["seqs"], 1)
    n = case["layers"] // 4
    return {k: n * a[k] + 3 * n * l[k] for k in a}


def tolerance(case):
    kind = case["kind"]
    if kind == "proj" and MIXES[case["mix"]][0] not in (Q8_0, BF16):
        # integer dots and block terms added in the order that the format's row dot defines: the same bits; a linear
        # layer's two small matrices in 32 bits aside
        return {"rel": 2e-6, "max": 1e-5, "differ": 0.0} if case["layer"] == "linear" else "exact"
    if kind == "proj":
        return {"rel": 4e-6, "max": 4e-5}
    if kind == "prefill":
        # products of bf16 pairs, 16 bits of each operand
        return {"rel": 4e-5, "max": 1e-3}
    if kind == "linear" and case["tokens"] > 1:
        return {"rel": 4e-5, "max": 1e-3}
    return {"rel": 2e-6, "max": 5e-5}


# ------------------------------------------------------------------ the same in 64 bits


def _sigmoid(x):
    return 1.0 / (1.0 + torch.exp(-x))


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _rope(x, positions):
    """x [n][heads][256]; the angle is the position times the scale, product by product in 32 bits, as the model defines it."""
    scale = np.float32(np.float32(10000000.0) ** np.float32(-2.0 / 64.0))
    theta, rows = np.array(positions, np.float32), []
    for _ in range(32):
        rows.append(theta.astype(np.float64))
        theta = (theta * scale).astype(np.float32)
    t = torch.from_numpy(np.stack(rows, 1)).to(x.device)[:, None, :]
    c, s, a, b = torch.cos(t), torch.sin(t), x[..., :32], x[..., 32:64]
    return torch.cat((a * c - b * s, a * s + b * c, x[..., 64:]), -1)


def _exact_decode(x, ks, vs, ctxs):
    qg = x["qg"].double().view(-1, HEADS, 2, HEAD_DIM)
    pos = [c - 1 for c in ctxs]
    q = _rope(_rms(qg[:, :, 0], x["q_norm"].double()), pos)
    k_new = _rope(_rms(x["key"].double().view(-1, KV_HEADS, HEAD_DIM), x["k_norm"].double()), pos)
    out = []
    for i, (k, v) in enumerate(zip(ks, vs)):
        k = torch.cat((k.double().view(-1, KV_HEADS, HEAD_DIM), k_new[i:i + 1]))
        v = torch.cat((v.double().view(-1, KV_HEADS, HEAD_DIM), x["value"][i:i + 1].double().view(1, KV_HEADS, HEAD_DIM)))
        heads = []
        for h in range(HEADS):
            p = torch.softmax(k[:, h // 6].contiguous() @ q[i, h] / 16.0, 0)
            heads.append(p @ v[:, h // 6].contiguous())
        out.append((torch.stack(heads) * _sigmoid(qg[i, :, 1])).reshape(-1))
    return torch.stack(out)


def _exact_linear(x, seqs, tokens):
    w, d = x["conv_w"].double(), {k: v.double() for k, v in x.items()}
    raw = d["qkv"].view(seqs, tokens, QKV_DIM)
    ext = torch.cat((d["conv"].permute(0, 2, 1), raw), 1)  # [seq][3 + tokens][channel]
    c = sum(ext[:, j:j + tokens] * w[:, j] for j in range(4))
    c = c * _sigmoid(c)
    conv = ext[:, tokens:].permute(0, 2, 1).contiguous()

    def unit(v):
        return v / torch.sqrt((v * v).sum(-1, keepdim=True)).clamp_min(1e-6)

    tile = torch.arange(LIN_V, device=c.device) % LIN_QK
    q = unit(c[..., :2048].reshape(seqs, tokens, LIN_QK, LIN_DIM))[:, :, tile] / math.sqrt(LIN_DIM)
    k = unit(c[..., 2048:4096].reshape(seqs, tokens, LIN_QK, LIN_DIM))[:, :, tile]
    v = c[..., 4096:].reshape(seqs, tokens, LIN_V, LIN_DIM)
    beta = _sigmoid(d["beta"]).view(seqs, tokens, LIN_V)
    decay = torch.exp(d["a"] * torch.nn.functional.softplus(d["alpha"] + d["dt"], threshold=40.0)).view(seqs, tokens, LIN_V)
    state, o = d["delta"].clone(), torch.empty_like(v)
    for t in range(tokens):
        state *= decay[:, t, :, None, None]
        kt = k[:, t, :, None, :]
        u = (v[:, t] - (state * kt).sum(-1)) * beta[:, t, :, None]
        state += u[..., None] * kt
        o[:, t] = (state * q[:, t, :, None, :]).sum(-1)
    z = d["z"].view(seqs, tokens, LIN_V, LIN_DIM)
    out = _rms(o, d["norm"]) * z * _sigmoid(z)
    return {"out": out.view(seqs * tokens, Q_DIM), "conv": conv, "delta": state}


def _grid(name):
    """A lattice grid of the IQ formats: [entries][4 or 8]; the formats define no rule for it but the table."""
    if name not in _held:
        with open(os.path.join(PKG_DIR, "csrc", "q38_iq_grids.h")) as f:
            body = re.search(r"#define %s \{(.*?)\}" % name, f.read(), re.S).group(1)
        vals = np.array([int(v, 16) for v in re.findall(r"0x[0-9a-f]+", body)], np.uint64)
        wide = 4 if "IQ3" in name else 8
        _held[name] = torch.from_numpy(vals.astype("<u8").view(np.uint8).reshape(-1, 8)[:, :wide].astype(np.float64)).cuda()
    return _held[name]


def _f16(b):
    return b.contiguous().view(torch.float16).double()


def _dequantised(ty, w, rows, width):
    """Rows of a format as 64-bit numbers."""
    if ty in (F32, BF16):
        return w.double()
    n = w.shape[0]
    b = w.to(torch.int32)
    lo4, hi4 = (lambda x: x & 15), (lambda x: x >> 4)  # noqa: E731
    if ty == Q8_0:
        v = _f16(w[:, :2]) * w[:, 2:].contiguous().view(torch.int8).double()
    elif ty in (12, 13):
        d, dmin, s = _f16(w[:, 0:2]), _f16(w[:, 2:4]), b[:, 4:16]
        sc = torch.cat((s[:, 0:4] & 63, lo4(s[:, 8:12]) | (s[:, 0:4] >> 6) << 4), 1)
        mn = torch.cat((s[:, 4:8] & 63, hi4(s[:, 8:12]) | (s[:, 4:8] >> 6) << 4), 1)
        qs = b[:, -128:].view(n, 4, 32)
        q = torch.stack((lo4(qs), hi4(qs)), 2).view(n, 8, 32)
        if ty == 13:
            q = q + 16 * ((b[:, None, 16:48] >> torch.arange(8, device=b.device)[None, :, None]) & 1)
        v = d[..., None] * sc[..., None] * q - (dmin * mn)[..., None]
    elif ty == 14:
        ql, qh = b[:, :128].view(n, 2, 2, 32), b[:, 128:192].view(n, 2, 32)
        q = torch.stack([(lo4(ql[:, :, 0]) if k == 0 else lo4(ql[:, :, 1]) if k == 1 else hi4(ql[:, :, 0]) if k == 2 else hi4(ql[:, :, 1]))
                         | ((qh >> (2 * k)) & 3) << 4 for k in range(4)], 2) - 32
        sc = w[:, 192:208].contiguous().view(torch.int8).double()
        v = _f16(w[:, 208:210])[..., None] * sc[..., None] * q.reshape(n, 16, 16)
    elif ty in (10, 11):
        qs = b[:, 16:80] if ty == 10 else b[:, 32:96]
        q = torch.stack([(qs.view(n, 2, 32) >> (2 * k)) & 3 for k in range(4)], 2).reshape(n, 16, 16)
        if ty == 10:
            sc = b[:, :16]
            v = _f16(w[:, 80:82])[..., None] * lo4(sc)[..., None] * q - (_f16(w[:, 82:84]) * hi4(sc))[..., None]
        else:
            high = torch.stack([(b[:, :32] >> m) & 1 for m in range(8)], 1).reshape(n, 16, 16)
            s = b[:, 96:108]
            sc = torch.cat((lo4(s[:, :8]), hi4(s[:, :8])), 1) | torch.cat([(s[:, 8:12] >> (2 * k)) & 3 for k in range(4)], 1) << 4
            v = _f16(w[:, 108:110])[..., None] * (sc - 32)[..., None] * (q - 4 + 4 * high)
    elif ty == 23:
        code = torch.tensor(IQ4, device=b.device, dtype=torch.float64)
        sh, at = b[:, 2] | b[:, 3] << 8, torch.arange(8, device=b.device)
        sc = ((b[:, 4:8].repeat_interleave(2, 1) >> (4 * (at % 2))) & 15 | ((sh[:, None] >> (2 * at)) & 3) << 4) - 32
        qs = b[:, 8:].view(n, 8, 16)
        v = _f16(w[:, 0:2])[..., None] * sc[..., None] * code[torch.cat((lo4(qs), hi4(qs)), 2).long()]
    else:
        eight, l = torch.arange(8, device=b.device), torch.arange(4, device=b.device)
        if ty == 22:  # qs[32] | signs[32] | qh[8] | scales[8]
            idx = b[:, 2:34].view(n, 8, 4) | (b[:, 66:74, None] << (8 - 2 * l)) & 0x300
            sc = torch.stack((lo4(b[:, 74:82]), hi4(b[:, 74:82])), 2).repeat_interleave(2, 2)
            signs = 1 - 2 * ((b[:, 34:66].view(n, 8, 4, 1) >> eight) & 1)
            v = (_f16(w[:, 0:2])[..., None] * (0.5 + sc) * 0.25)[..., None] * _grid("Q38_IQ2S_GRID")[idx.long()] * signs
        else:  # IQ3_S: qs[64] | qh[8] | signs[32] | scales[4]
            qs, qh = b[:, 2:66].view(n, 8, 4, 2), b[:, 66:74, None]
            idx = torch.stack((qs[..., 0] | (qh << (8 - 2 * l)) & 256, qs[..., 1] | (qh << (7 - 2 * l)) & 256), -1)
            sc = torch.stack((lo4(b[:, 106:110]), hi4(b[:, 106:110])), 2).view(n, 8)
            signs = 1 - 2 * ((b[:, 74:106].view(n, 8, 4, 1) >> eight) & 1)
            v = (_f16(w[:, 0:2]) * (1 + 2 * sc))[..., None, None] * _grid("Q38_IQ3S_GRID")[idx.long()].view(n, 8, 4, 8) * signs
    return v.reshape(rows, width)


def _q8k(x):
    """The values that the 8-bit activations stand for: 256 share the scale of the one of largest size, which becomes -127."""
    v = x.view(-1, 256).double()
    m = v.gather(1, v.abs().argmax(1, keepdim=True))
    inv = torch.where(m == 0, 0.0, -127.0 / m)
    q = torch.round(v * inv).clamp_max(127.0)
    return (q * torch.where(m == 0, 0.0, m / -127.0)).view(x.shape)


def exact(case, seed):
    g, kind = _Gen(seed), case["kind"]
    if kind == "decode":
        ctxs = _contexts(case)
        x, ks, vs = _attention_inputs(g, len(ctxs)), [], []
        for c in ctxs:
            ks.append(g.normal(c - 1, KV_DIM))
            vs.append(g.normal(c - 1, KV_DIM))
        return _exact_decode(x, ks, vs, ctxs)
    if kind == "prefill":
        base, n = case["base"], case["tokens"]
        x = _prefill_inputs(g, base, n)
        out = torch.empty((n, HEADS, HEAD_DIM), device="cuda", dtype=torch.float64)
        late = torch.arange(base + n, device="cuda")[None, :] > torch.arange(base, base + n, device="cuda")[:, None]
        for h in range(HEADS):
            k = x["k"].view(-1, KV_HEADS, HEAD_DIM)[:, h // 6].double()
            v = x["v"].view(-1, KV_HEADS, HEAD_DIM)[:, h // 6].double().contiguous()
            s = x["q"].view(n, HEADS, HEAD_DIM)[:, h].double() @ k.t().contiguous() / 16.0
            out[:, h] = torch.softmax(s.masked_fill_(late, -math.inf), 1) @ v
        return (out.view(n, Q_DIM) * _sigmoid(x["gate"].double()))
    if kind == "linear":
        return _exact_linear(_linear_inputs(g, case["seqs"], case["tokens"]), case["seqs"], case["tokens"])
    if kind == "proj":
        result = []
        for ty, rows, width in _groups(case):
            ws = [_weights(g, ty, r, width) for r in rows]
            x = g.normal(case["tokens"], width)
            q8 = ty in BLOCKS and BLOCKS[ty][1] == 256
            a = _q8k(x) if q8 else x.double()
            outs = [a @ _dequantised(ty, w, r, width).t().contiguous() for w, r in zip(ws, rows)]
            result.append({"outs": outs, "q8k": None} if q8 else {"outs": outs})
        return result
    ctxs, outs, convs, deltas = _contexts(case), [], [], []
    for layer in range(case["layers"]):
        if layer % 4 == 3:
            x, ks, vs = _attention_inputs(g, len(ctxs)), [], []
            for c in ctxs:
                ks.append(g.normal(c - 1, KV_DIM))
                vs.append(g.normal(c - 1, KV_DIM))
            outs.append(_exact_decode(x, ks, vs, ctxs))
        else:
            e = _exact_linear(_linear_inputs(g, len(ctxs), 1), len(ctxs), 1)
            outs.append(e["out"])
            convs.append(e["conv"])
            deltas.append(e["delta"])
    return {"outs": torch.stack(outs), "conv": torch.stack(convs), "delta": torch.stack(deltas)}
