"""The work whose speed is followed: calls a language-model server makes of this library, from a single projection of
one decoded token to the MLP of a long prompt.

Each case is one pass through the public Python entry points of kriya_q4 on inputs and weights resident on the GPU.
Weights are uniform nibbles with bf16 scales and biases -7.5 * scale (rows of mean zero), scaled so that a projection
keeps the size of its input; activations are N(0, 1) with every 61st channel eight times larger, as the outlier channels of real models.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "kriya-rt_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import kriya_q4 as kq  # noqa: E402
from kriya_q4 import qwen_decode as qd  # noqa: E402

EPS = 1e-6
ROPE_THETA = 1e6
LARGEST_FLOPS = 5.5e11  # of the largest listed case; drawn ones stay below it
LARGEST_BYTES = 6e8

ACT = {"swiglu": kq.ACT_SWIGLU, "geglu": kq.ACT_GEGLU, "relu": kq.ACT_RELU}


def listed():
    return [
        # One decoded token's output projection: the smallest call, where the launch counts.
        {"name": "linear_m1", "kind": "linear", "m": 1, "n": 2048, "k": 2048, "out": "bf16", "acc": False, "ws": False},
        # The down projection of a small batch of sequences, called without a workspace: a long K, an odd row count.
        {"name": "linear_m27_long", "kind": "linear", "m": 27, "n": 2048, "k": 11008, "out": "f32", "acc": True,
         "ws": False},
        # Six consecutive MLP layers of single-stream decode (norm, gate/up, down, residual).
        {"name": "mlp_m1", "kind": "mlp", "m": 1, "hidden": 2048, "inter": 11008, "layers": 6, "act": "swiglu"},
        # MLP layers of a large decode batch (or a short prompt), not a round number of rows.
        {"name": "mlp_m100", "kind": "mlp", "m": 100, "hidden": 2048, "inter": 11008, "layers": 2, "act": "swiglu"},
        # Query, key and value projections of a 512-token prompt, with the norm before them and their biases.
        {"name": "qkv_m512", "kind": "qkv", "m": 512, "hidden": 2048, "q_heads": 16, "kv_heads": 2, "head_dim": 128},
        # The MLP of a 512-token prompt.
        {"name": "mlp_m512", "kind": "mlp", "m": 512, "hidden": 2048, "inter": 11008, "layers": 1, "act": "swiglu"},
        # The MLP of a long prompt (the largest case): 3907 tokens, a ragged last tile.
        {"name": "mlp_m3907", "kind": "mlp", "m": 3907, "hidden": 2048, "inter": 11008, "layers": 1, "act": "swiglu"},
        # The attention half of a decode layer for five sequences of different lengths up to 3000 positions.
        {"name": "attn_b5", "kind": "attn", "m": 5, "ctx": 3000, "hidden": 2048, "q_heads": 16, "kv_heads": 2,
         "head_dim": 128},
        # Routed experts of one decoded token, of a decode batch of 64 and of a 1000-token prompt.
        {"name": "moe_t1", "kind": "moe", "m": 1, "experts": 60, "topk": 4, "hidden": 2048, "inter": 1408,
         "out": "bf16"},
        {"name": "moe_t64", "kind": "moe", "m": 64, "experts": 60, "topk": 4, "hidden": 2048, "inter": 1408,
         "out": "bf16"},
        {"name": "moe_t1000", "kind": "moe", "m": 1000, "experts": 60, "topk": 4, "hidden": 2048, "inter": 1408,
         "out": "bf16"},
        # A whole decode step of 16 sequences: embedding, eight layers, norm and the vocabulary's logits.
        {"name": "decoder_b16", "kind": "decoder", "m": 16, "ctx": 512, "layers": 8},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng):
    """Token rows as they occur: few while decoding, any number up to a long prompt's while prefilling."""
    return rng.choice([1, _log_int(rng, 2, 16), _log_int(rng, 5, 64), _log_int(rng, 33, 512), _log_int(rng, 128, 4096)])


def draw(rng):
    while True:
        kind = rng.choice(["linear", "linear", "mlp", "mlp", "mlp", "qkv", "attn", "moe", "moe", "decoder"])
        if kind == "linear":
            case = {"kind": kind, "m": _rows(rng), "n": rng.choice([_log_int(rng, 1000, 16384), 8 * rng.randint(64, 2048)]),
                    "k": 64 * _log_int(rng, 12, 296), "out": rng.choice(["bf16", "f32"]),
                    "acc": rng.random() < 0.5, "ws": rng.random() < 0.5}
        elif kind == "mlp":
            hidden = 64 * rng.choice([16, 24, 28, 32, 32, 40, 48, 56, 64])
            m = _rows(rng)
            case = {"kind": kind, "m": m, "hidden": hidden, "inter": 64 * max(12, int(hidden / 64 * rng.uniform(1.3, 5.6))),
                    "layers": 4 if m <= 16 else 1, "act": rng.choice(["swiglu", "swiglu", "swiglu", "geglu", "relu"])}
        elif kind == "qkv":
            kv = rng.choice([1, 2, 4, 8])
            case = {"kind": kind, "m": _rows(rng), "hidden": 64 * rng.choice([16, 24, 32, 40, 56, 64]),
                    "q_heads": kv * rng.randint(1, 8), "kv_heads": kv, "head_dim": rng.choice([64, 128])}
        elif kind == "attn":
            kv = rng.choice([1, 2, 4, 8])
            case = {"kind": kind, "m": _log_int(rng, 1, 32), "ctx": _log_int(rng, 64, 8000),
                    "hidden": 64 * rng.choice([16, 24, 32, 40]), "q_heads": kv * rng.randint(1, 8), "kv_heads": kv,
                    "head_dim": rng.choice([64, 128, 128])}
        elif kind == "moe":
            experts = rng.choice([8, 16, 32, 60, 64, 128])
            case = {"kind": kind, "m": rng.choice([_log_int(rng, 1, 8), _log_int(rng, 5, 200), _log_int(rng, 100, 2000)]),
                    "experts": experts, "topk": rng.randint(1, 8), "hidden": 128 * rng.randint(8, 16),
                    "inter": 128 * rng.randint(4, 16), "out": rng.choice(["bf16", "f32"])}
        else:
            case = {"kind": kind, "m": _log_int(rng, 1, 32), "ctx": _log_int(rng, 32, 2000), "layers": rng.randint(2, 8)}
        w = work(case)
        if w["flops"] <= LARGEST_FLOPS and w["bytes"] <= LARGEST_BYTES:
            return case


# ---- inputs ------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _q4(n, k, g, gain=1.0):
    """Q4_G64 weights whose rows have a 2-norm of about `gain` (uniform nibbles minus 7.5 have a root mean square of 4.61)."""
    qw = torch.randint(-(2 ** 31), 2 ** 31 - 1, (n, k // 8), dtype=torch.int32, device="cuda", generator=g)
    s = ((0.6 + 0.4 * torch.randn((n, k // 64), device="cuda", generator=g).abs()) * (gain / 4.61 / math.sqrt(k)))
    s = s.to(torch.bfloat16)
    return kq.Q4Matrix(qw, s.view(torch.int16), (s.float() * -7.5).to(torch.bfloat16).view(torch.int16))


def _x(m, k, g, gain=1.0):
    x = torch.randn((m, k), device="cuda", generator=g) * gain
    x[:, ::61] *= 8.0
    return x.to(torch.bfloat16)


def _vec(n, g, mean=0.0, dev=0.1):
    return (mean + dev * torch.randn(n, device="cuda", generator=g)).to(torch.bfloat16)


def _positions(case, g):
    """One position per sequence, from half of the longest context up; the first has the longest."""
    p = torch.randint(case["ctx"] // 2, case["ctx"], (case["m"],), device="cuda", generator=g, dtype=torch.int32)
    p[0] = case["ctx"] - 1
    return p


def _dt(case):
    return torch.float32 if case["out"] == "f32" else torch.bfloat16


def prepare(case, seed):
    g, m, kind = _gen(seed), case["m"], case["kind"]
    s = {"case": case}
    if kind == "linear":
        s["w"], s["x"] = _q4(case["n"], case["k"], g), _x(m, case["k"], g)
        s["y0"] = torch.randn((m, case["n"]), device="cuda", generator=g).to(_dt(case))
        s["y"] = s["y0"].clone()
        s["workspace"] = kq.linear_workspace(m, case["n"], case["k"]) if case["ws"] else None
    elif kind == "mlp":
        hidden, inter = case["hidden"], case["inter"]
        s["layers"] = [(_q4(inter, hidden, g), _q4(inter, hidden, g), _q4(hidden, inter, g), _vec(hidden, g, 1.0))
                       for _ in range(case["layers"])]
        s["h0"] = _x(m, hidden, g)
        s["h"] = s["h0"].clone()
        s["workspace"] = kq.rmsnorm_mlp_workspace(m, hidden, inter)
    elif kind in ("qkv", "attn"):
        hidden, qn, kn = case["hidden"], case["q_heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        s["w"] = tuple(_q4(n, hidden, g) for n in (qn, kn, kn))
        s["b"] = tuple(_vec(n, g) for n in (qn, kn, kn))
        s["ln"] = _vec(hidden, g, 1.0)
        s["h"] = _x(m, hidden, g)
        s["outs"] = tuple(torch.empty((m, n), dtype=torch.bfloat16, device="cuda") for n in (qn, kn, kn))
        s["xnorm"] = torch.empty((m, hidden), dtype=torch.bfloat16, device="cuda")
        if kind == "attn":
            s["o"] = _q4(hidden, qn, g)
            s["h0"] = s["h"].clone()
            s["pos"] = _positions(case, g)
            s["cos_sin"] = qd.rope_table(case["ctx"], case["head_dim"], ROPE_THETA).cuda()
            shape = (m, case["ctx"], case["kv_heads"], case["head_dim"])
            s["k_cache"] = torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)
            s["v_cache"] = torch.randn(shape, device="cuda", generator=g).to(torch.bfloat16)
            s["workspace"] = kq.attention_q4_out_workspace(m, case["q_heads"], case["head_dim"], case["ctx"])
    elif kind == "moe":
        e, hidden, inter = case["experts"], case["hidden"], case["inter"]
        s["w"] = (_q4(e * inter, hidden, g), _q4(e * inter, hidden, g), _q4(e * hidden, inter, g))
        s["x"] = _x(m, hidden, g)
        s["logits"] = torch.randn((m, e), device="cuda", generator=g)
        s["route"] = kq.MoeRoute(m, e, case["topk"])
        s["y"] = torch.empty((m, hidden), dtype=_dt(case), device="cuda")
        s["workspace"] = kq.moe_workspace(m, case["topk"], hidden, inter)
    else:
        dec = qd.QwenQ4Decoder(qd.QwenConfig(layers=case["layers"]), batch=m, ctx=case["ctx"], seed=seed)
        for L in dec.layers:  # an eighth of the decoder's own random weights keeps each layer's output at its input's size
            for w in (L.q, L.k, L.v, L.o, L.gate, L.up, L.down):
                w.scales.view(torch.bfloat16).mul_(0.125)
                w.biases.view(torch.bfloat16).mul_(0.125)
        s["dec"], s["tokens"] = dec, dec.tokens.clone()
    return s


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "linear":
        if case["acc"]:
            s["y"].copy_(s["y0"])
        return kq.q4_linear(s["w"], s["x"], y=s["y"], accumulate=case["acc"], workspace=s["workspace"])
    if kind == "mlp":
        h = s["h"]
        h.copy_(s["h0"])
        for gate, up, down, ln in s["layers"]:
            kq.rmsnorm_mlp(gate, up, down, h, ln, EPS, activation=ACT[case["act"]], workspace=s["workspace"])
        return h
    if kind == "qkv":
        return kq.rmsnorm_qkv(s["h"], s["ln"], EPS, *s["w"], *s["b"], outs=s["outs"], xnorm=s["xnorm"])
    if kind == "attn":
        h = s["h"]
        h.copy_(s["h0"])
        q, k, v = kq.rmsnorm_qkv(h, s["ln"], EPS, *s["w"], *s["b"], outs=s["outs"], xnorm=s["xnorm"])
        kq.rope_attention_q4_out(q, k, v, s["cos_sin"], s["pos"], case["q_heads"], case["kv_heads"], case["head_dim"],
                                 s["k_cache"], s["v_cache"], s["o"], h, workspace=s["workspace"])
        return h, s["k_cache"], s["v_cache"]
    if kind == "moe":
        y, route = kq.moe_route_experts(*s["w"], case["experts"], s["x"], s["logits"], case["topk"], out=s["route"],
                                        y=s["y"], workspace=s["workspace"])
        return y, route.selected, route.weights
    dec = s["dec"]
    dec.tokens.copy_(s["tokens"])
    dec.step()
    return dec.logits


# ---- what a pass cannot do without ---------------------------------------------------------

def _q4_bytes(n, k):
    return n * k // 2 + n * (k // 64) * 4


def work(case):
    m, kind = case["m"], case["kind"]
    if kind == "linear":
        n, k = case["n"], case["k"]
        out = m * n * (4 if case["out"] == "f32" else 2)
        return {"bytes": _q4_bytes(n, k) + 2 * m * k + out * (2 if case["acc"] else 1), "flops": 2 * m * n * k}
    if kind == "mlp":
        h, i, layers = case["hidden"], case["inter"], case["layers"]
        return {"bytes": layers * (2 * _q4_bytes(i, h) + _q4_bytes(h, i)) + 4 * m * h, "flops": layers * 6 * m * h * i}
    if kind in ("qkv", "attn"):
        h, d = case["hidden"], case["head_dim"]
        qn, kn = case["q_heads"] * d, case["kv_heads"] * d
        n = qn + 2 * kn
        b, f = _q4_bytes(n, h) + 2 * m * (h + n), 2 * m * n * h
        if kind == "attn":
            rows = m * 0.75 * case["ctx"]  # the positions of an average draw
            b += int(rows * 2 * kn * 2) + _q4_bytes(h, qn) + 2 * m * h
            f += 2 * m * qn * h + int(4 * rows * qn)
        return {"bytes": b, "flops": f}
    if kind == "moe":
        h, i, e, a = case["hidden"], case["inter"], case["experts"], m * min(case["topk"], case["experts"])
        hit = e * (1.0 - (1.0 - a / m / e) ** m)  # experts that an average routing reaches
        return {"bytes": int(hit * (2 * _q4_bytes(i, h) + _q4_bytes(h, i))) + m * h * (2 + (4 if case["out"] == "f32" else 2)),
                "flops": 6 * a * h * i}
    c = qd.QwenConfig(layers=case["layers"])
    b = c.q4_bytes_per_step()
    kv = 2 * c.layers * m * case["ctx"] * c.kv_heads * c.head_dim * 2
    attn = 4 * c.layers * m * case["ctx"] * c.q_heads * c.head_dim
    return {"bytes": b + kv + 4 * m * c.vocab, "flops": int(2 * m * b / 0.5625) + attn}


def tolerance(case):
    """About four times the distance from the 64-bit result: one or two bf16 roundings (1.7e-3 to 2.3e-3) on every
    path with bf16 outputs or intermediates, f32 summation for the f32 linear of few rows, fp16 weights above."""
    if case["kind"] == "linear" and case["out"] == "f32":
        return {"rel": 1e-3} if case["m"] >= 64 else {"rel": 2e-6}
    if case["kind"] == "decoder":
        return {"rel": 5e-3}  # measured 1.0e-3: the logits are mostly the embedding's
    if case["kind"] == "mlp" and case["layers"] > 1:
        return {"rel": 1.6e-2}  # a single row's bf16 roundings through several layers: up to 5.4e-3
    return {"rel": 8e-3}


# ---- the same in 64 bits -------------------------------------------------------------------

def _w64(w, lo=0, hi=None):
    """Rows lo .. hi of a planar Q4_G64 matrix, dequantised in 64 bits."""
    hi = w.n if hi is None else hi
    shifts = torch.arange(0, 32, 4, dtype=torch.int32, device="cuda")
    q = ((w.qw[lo:hi].unsqueeze(-1) >> shifts) & 15).double().view(hi - lo, w.k // 64, 64)
    s = w.scales[lo:hi].view(torch.bfloat16).double().unsqueeze(-1)
    b = w.biases[lo:hi].view(torch.bfloat16).double().unsqueeze(-1)
    return (q * s + b).view(hi - lo, w.k)


def _mul64(x, w, lo=0, hi=None):
    return x @ _w64(w, lo, hi).t()


def _norm64(x, ln):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * ln.double()


def _act64(g, act):
    if act == "swiglu":
        return g * torch.sigmoid(g)
    if act == "geglu":
        return torch.nn.functional.gelu(g, approximate="tanh")
    return torch.relu(g)


def _attn64(q, k, v, cos_sin, pos, heads, kv_heads, d, k_cache, v_cache):
    """(attention's result, the caches with the new rows) for one token per sequence."""
    m = pos.numel()
    rows = torch.arange(m, device="cuda")
    cs = cos_sin.double()[pos.long()].unsqueeze(1)

    def rope(t):
        a, b = t[..., : d // 2], t[..., d // 2:]
        return torch.cat([a * cs[..., 0] - b * cs[..., 1], a * cs[..., 1] + b * cs[..., 0]], -1)

    q, k, v = rope(q.view(m, heads, d)), rope(k.view(m, kv_heads, d)), v.view(m, kv_heads, d)
    kc, vc = k_cache.double(), v_cache.double()
    kc[rows, pos.long()], vc[rows, pos.long()] = k, v
    out = torch.empty((m, heads, d), dtype=torch.float64, device="cuda")
    for b in range(m):
        n = int(pos[b]) + 1
        for j in range(kv_heads):
            hs = slice(j * (heads // kv_heads), (j + 1) * (heads // kv_heads))
            p = torch.softmax(q[b, hs] @ kc[b, :n, j].t() / math.sqrt(d), -1)
            out[b, hs] = p @ vc[b, :n, j]
    return out.view(m, heads * d), kc, vc


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind == "linear":
        y = _mul64(s["x"].double(), s["w"])
        return s["y0"].double() + y if case["acc"] else y
    if kind == "mlp":
        h = s["h0"].double()
        for gate, up, down, ln in s["layers"]:
            x = _norm64(h, ln)
            h = h + _mul64(_act64(_mul64(x, gate), case["act"]) * _mul64(x, up), down)
        return h
    if kind in ("qkv", "attn"):
        x = _norm64(s["h"].double(), s["ln"])
        q, k, v = (_mul64(x, w) + b.double() for w, b in zip(s["w"], s["b"]))
        if kind == "qkv":
            return q, k, v
        a, kc, vc = _attn64(q, k, v, s["cos_sin"], s["pos"], case["q_heads"], case["kv_heads"], case["head_dim"],
                            s["k_cache"], s["v_cache"])
        return s["h"].double() + _mul64(a, s["o"]), kc, vc
    if kind == "moe":
        gate, up, down = s["w"]
        hidden, inter, x = case["hidden"], case["inter"], s["x"].double()
        p, ids = torch.softmax(s["logits"].double(), -1).topk(min(case["topk"], case["experts"]), -1)
        p = p / p.sum(-1, keepdim=True)
        y = torch.zeros((case["m"], hidden), dtype=torch.float64, device="cuda")
        for e in range(case["experts"]):
            t, slot = torch.nonzero(ids == e, as_tuple=True)
            if t.numel():
                a = _act64(_mul64(x[t], gate, e * inter, (e + 1) * inter), "swiglu")
                a = a * _mul64(x[t], up, e * inter, (e + 1) * inter)
                y.index_add_(0, t, _mul64(a, down, e * hidden, (e + 1) * hidden) * p[t, slot].unsqueeze(-1))
        return y, None, p
    dec, c = s["dec"], s["dec"].cfg
    h = _w64_rows(dec.embed, s["tokens"])
    for L in dec.layers:
        x = _norm64(h, L.ln1)
        q, k, v = (_mul64(x, w) + b.double() for w, b in ((L.q, L.bq), (L.k, L.bk), (L.v, L.bv)))
        a, _, _ = _attn64(q, k, v, dec.cos_sin, dec.positions, c.q_heads, c.kv_heads, c.head_dim, L.k_cache, L.v_cache)
        h = h + _mul64(a, L.o)
        x = _norm64(h, L.ln2)
        h = h + _mul64(_act64(_mul64(x, L.gate), "swiglu") * _mul64(x, L.up), L.down)
    return _mul64(_norm64(h, dec.ln_f), dec.embed)


def _w64_rows(w, ids):
    i = ids.long()
    return _w64(kq.Q4Matrix(w.qw[i].contiguous(), w.scales[i].contiguous(), w.biases[i].contiguous()))
