"""The work that a user of this library has it do, as timed cases.

Each case goes through the public Python operators (clef-hrx_amd/clef_i4.py)
as a model's forward pass or its loader calls them: the activation comes in as
bf16 and is quantized by the call, the packed weights are resident. Sizes are
those of the repository's benchmark, tests and published token counts: dense
widths 4096/12288 and 5120/17408, the Omni MoE block (hidden 2048, 128 experts,
top-8, expert width 768), and 235, 620 and 2729 prompt tokens.

Integer dot products are exact and every rounding step of the outputs is part
of the operators' definition, so a correct change of the code changes no bit:
every tolerance is "exact". exact() is the same function in float64, with the
bf16 tensors that the path materializes rounded to bf16.
"""
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "clef-hrx_amd"))

import clef_i4  # noqa: E402

EXPERTS = 128


def listed():
    return [
        # One decoded token through a projection of the default resident form
        # (INT4 codes): latency and the weight stream are the whole cost.
        {"name": "linear_int4_m1", "kind": "linear", "form": "int4", "m": 1, "k": 4096, "n": 12288,
         "residual": False},
        # The single linear of the reference's own CPU-path benchmark.
        {"name": "linear_int4_m512", "kind": "linear", "form": "int4", "m": 512, "k": 2048, "n": 2048,
         "residual": False},
        # A batch of 37 decode streams, output projection with its residual,
        # weights kept in the bf6 form alone.
        {"name": "linear_bf6_m37_res", "kind": "linear", "form": "bf6", "m": 37, "k": 4096, "n": 4096,
         "residual": True},
        # The 8-bit packing of a projection over a 235-token prompt.
        {"name": "linear_int8_m235", "kind": "linear", "form": "int8", "m": 235, "k": 4096, "n": 12288,
         "residual": False},
        # Fused-norm INT4 MLP block over a 2729-token prompt, default form.
        {"name": "mlp_int4_m2729", "kind": "mlp", "form": "int4", "norm": True, "m": 2729, "d": 5120, "f": 17408},
        # The same model's MLP on the bf6 form over a 620-token prompt.
        {"name": "mlp_bf6_m620", "kind": "mlp", "form": "bf6", "norm": False, "m": 620, "d": 5120, "f": 17408},
        # The benchmark's MLP block: a full prefill chunk.
        {"name": "mlp_bf6_m4096", "kind": "mlp", "form": "bf6", "norm": False, "m": 4096, "d": 4096, "f": 12288},
        # Omni MoE block, hidden states in, router gate included: one decoded
        # token, a 235-token prompt, a full prefill chunk.
        {"name": "moe_t1", "kind": "moe", "t": 1, "d": 2048, "f": 768, "topk": 8, "router": True, "skewed": False},
        {"name": "moe_t235", "kind": "moe", "t": 235, "d": 2048, "f": 768, "topk": 8, "router": True,
         "skewed": False},
        {"name": "moe_t4096", "kind": "moe", "t": 4096, "d": 2048, "f": 768, "topk": 8, "router": True,
         "skewed": False},
        # A packed batch of long prompts whose routing is skewed (one expert
        # with tens of thousands of rows, eight with none), logits given.
        {"name": "moe_t65536_skewed", "kind": "moe", "t": 65536, "d": 2048, "f": 768, "topk": 8, "router": False,
         "skewed": True},
        # Loading one projection of a tiled checkpoint: packed to INT4 codes
        # and re-encoded as bf6, both kept.
        {"name": "load_int4_bf6", "kind": "load", "rows": 12288, "cols": 4096, "bits": 4, "tiled": True, "bf6": True},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mult(rng, lo, hi, step):
    """A multiple of `step`, log-uniform in [lo, hi]."""
    return max(lo, min(hi, round(_log(rng, lo, hi) / step) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "mlp", "moe", "moe", "attention", "load"])
    if kind == "linear":
        return {"kind": kind, "form": rng.choice(["int4", "bf6", "int8"]), "m": _log(rng, 1, 8192),
                "k": _mult(rng, 1024, 12288, 256), "n": _mult(rng, 1024, 12288, 256),
                "residual": rng.random() < 0.4}
    if kind == "mlp":
        norm = rng.random() < 0.5
        return {"kind": kind, "form": "int4" if norm else "bf6", "norm": norm, "m": _log(rng, 1, 4096),
                "d": 5120 if norm else _mult(rng, 2048, 5120, 256), "f": _mult(rng, 4096, 17408, 256)}
    if kind == "moe":
        t = _log(rng, 1, 16384)
        return {"kind": kind, "t": t, "d": 2048, "f": 768, "topk": 8, "router": rng.random() < 0.7,
                "skewed": False} if rng.random() < 0.6 else \
               {"kind": kind, "t": t, "d": _mult(rng, 1024, 2048, 256), "f": _mult(rng, 512, 1024, 256),
                "topk": rng.choice([4, 6, 8]), "router": False, "skewed": True}
    if kind == "attention":
        # attention block of the 5120-wide model: norm-fused q|gate, k and v
        # projections, then the gated output projection with its residual
        return {"kind": kind, "m": _log(rng, 1, 4096), "d": 5120, "width": _mult(rng, 4096, 6144, 512),
                "kv": 1024, "bits": rng.choice([4, 4, 8])}
    return {"kind": kind, "rows": _mult(rng, 4096, 24576, 256), "cols": _mult(rng, 1024, 8192, 256),
            "bits": rng.choice([4, 4, 8]), "tiled": rng.random() < 0.7, "bf6": False}


# ---------------------------------------------------------------- inputs

class _Gen:
    """Seeded tensors of one state: activations N(0,1), weights N(0,0.02)."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + 17)

    def randn(self, shape, std=1.0):
        x = torch.randn(shape, generator=self.g, device="cuda", dtype=torch.bfloat16)
        return x if std == 1.0 else x.mul_(std)

    def f32(self, shape):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32)


def _raw(case, seed):
    """The bf16 tensors a case starts from, made from the seed alone."""
    g = _Gen(seed)
    kind = case["kind"]
    if kind == "linear":
        r = {"x": g.randn((case["m"], case["k"])), "w": g.randn((case["n"], case["k"]), 0.02)}
        r["res"] = g.randn((case["m"], case["n"])) if case["residual"] else None
        return r
    if kind == "mlp":
        r = {"x": g.randn((case["m"], case["d"])), "gate": g.randn((case["f"], case["d"]), 0.02),
             "up": g.randn((case["f"], case["d"]), 0.02), "down": g.randn((case["d"], case["f"]), 0.02)}
        r["nw"] = g.randn((case["d"],), 0.1) if case["norm"] else None
        return r
    if kind == "attention":
        m, d, w, kv = case["m"], case["d"], case["width"], case["kv"]
        return {"x": g.randn((m, d)), "nw": g.randn((d,), 0.1), "q": g.randn((2 * w, d), 0.02),
                "k": g.randn((kv, d), 0.02), "v": g.randn((kv, d), 0.02), "o": g.randn((d, w), 0.02),
                # attention itself is another library's: its output stands for it
                "att": g.randn((m, w))}
    if kind == "moe":
        t, d, f = case["t"], case["d"], case["f"]
        r = {"x": g.randn((t, d)), "gate": g.randn((EXPERTS * f, d), 0.02), "up": g.randn((EXPERTS * f, d), 0.02),
             "down": g.randn((EXPERTS * d, f), 0.02), "router": None, "logits": None}
        if case["router"]:
            r["router"] = g.randn((EXPERTS, d), 0.02)
        else:
            z = g.f32((t, EXPERTS))
            if case["skewed"]:
                # Zipf-like popularity; the eight least popular are never chosen
                rank = torch.randperm(EXPERTS, generator=g.g, device="cuda").float()
                bias = -1.1 * 0.57 * torch.log1p(rank)
                z = z + torch.where(rank >= EXPERTS - 8, torch.full_like(bias, -30.0), bias)
            r["logits"] = z.to(torch.bfloat16)
        return r
    return {"w": g.randn((case["rows"], case["cols"]), 0.02)}


def _pack(w, form):
    q = clef_i4.load_quantized_weight(w, bits=8 if form == "int8" else 4)
    return clef_i4.f6_weight(q) if form == "bf6" else q


def prepare(case, seed):
    r = _raw(case, seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        s.update(x=r["x"], res=r["res"], w=_pack(r["w"], case["form"]))
    elif kind == "mlp":
        s.update(x=r["x"], nw=r["nw"], **{n: _pack(r[n], case["form"]) for n in ("gate", "up", "down")})
    elif kind == "attention":
        form = "int8" if case["bits"] == 8 else "int4"
        s.update(x=r["x"], nw=r["nw"], att=r["att"], **{n: _pack(r[n], form) for n in ("q", "k", "v", "o")})
    elif kind == "moe":
        s.update(x=r["x"], logits=r["logits"],
                 layer=clef_i4.MoeLayer(*(_pack(r[n], "int4") for n in ("gate", "up", "down")), topk=case["topk"],
                                        router=r["router"]))
    else:
        s.update(w=r["w"])
    return s


# ---------------------------------------------------------------- one pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["form"] == "bf6":
            return clef_i4.project_quantized_f6(state["x"], state["w"], state["res"])
        if case["form"] == "int4":
            return clef_i4.project_quantized(state["x"], state["w"], state["res"])
        return clef_i4.project_prepared(clef_i4.prepare(state["x"], bits=8), state["w"], residual=state["res"])
    if kind == "mlp":
        gate, up, down = state["gate"], state["up"], state["down"]
        if case["form"] == "bf6":
            h = clef_i4.project_gate_up_f6(clef_i4.prepare_f6(state["x"]), gate, up)
            return clef_i4.project_f6(clef_i4.prepare_f6(h), down, residual=state["x"])
        if case["norm"]:
            a, _ = clef_i4.prepare_norm(state["x"], state["nw"])
        else:
            a = clef_i4.prepare(state["x"])
        g, u = clef_i4.project_prepared(a, gate), clef_i4.project_prepared(a, up)
        return clef_i4.project_prepared(clef_i4.prepare_swiglu(g, u), down, residual=state["x"])
    if kind == "attention":
        a, _ = clef_i4.prepare_norm(state["x"], state["nw"], bits=case["bits"])
        q, k, v = (clef_i4.project_prepared(a, state[n]) for n in ("q", "k", "v"))
        return q, k, v, clef_i4.project_attention_gate(state["att"], q, state["o"], state["x"])
    if kind == "moe":
        return state["layer"](state["x"], state["logits"])
    w = clef_i4.load_quantized_weight(state["w"], bits=case["bits"], tiled_checkpoint=case["tiled"])
    if case["bf6"]:
        return w.codes, w.scales, clef_i4.f6_weight(w).codes
    return w.codes, w.scales


# ---------------------------------------------------------------- floors

def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        wb = {"int4": 0.5, "bf6": 0.75, "int8": 1.0}[case["form"]]
        return {"bytes": 2 * m * k + wb * n * k + 4 * n + 2 * m * n * (2 if case["residual"] else 1),
                "flops": 2.0 * m * n * k}
    if kind == "mlp":
        m, d, f = case["m"], case["d"], case["f"]
        wb = 0.75 if case["form"] == "bf6" else 0.5
        return {"bytes": 4 * m * d + wb * 3 * d * f + 4 * (2 * f + d), "flops": 6.0 * m * d * f}
    if kind == "attention":
        m, d, w, kv = case["m"], case["d"], case["width"], case["kv"]
        wb = case["bits"] / 8
        cols = d * (3 * w + 2 * kv)
        return {"bytes": 4 * m * d + 2 * m * (3 * w + 2 * kv) + wb * cols + 4 * (2 * w + 2 * kv + d),
                "flops": 2.0 * m * cols}
    if kind == "moe":
        t, d, f, topk = case["t"], case["d"], case["f"], case["topk"]
        live = EXPERTS - 8 if case["skewed"] else EXPERTS
        # experts that t tokens of evenly spread routes reach
        active = live * (1.0 - (1.0 - topk / live) ** t)
        return {"bytes": active * (1.5 * f * d + 4 * (2 * f + d)) + 4 * t * d
                + (2 * EXPERTS * d if case["router"] else 2 * EXPERTS * t),
                "flops": 6.0 * t * topk * f * d + (2.0 * t * EXPERTS * d if case["router"] else 0.0)}
    r, c = case["rows"], case["cols"]
    out = case["bits"] / 8 + (0.75 if case["bf6"] else 0.0)
    return {"bytes": r * c * (2 + out) + 4 * r, "flops": 16.0 * r * c}


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------- float64

def _had(dev):
    h = torch.tensor([[1, 1, 1, -1], [1, 1, -1, 1], [1, -1, 1, 1], [-1, 1, 1, 1]], dtype=torch.float64, device=dev)
    k = torch.ones((1, 1), dtype=torch.float64, device=dev)
    for _ in range(4):
        k = torch.kron(h, k)
    return k


def _quant(x, bits=4):
    """Rotated per-row quantizer in float64: (codes, scales)."""
    rows, width = x.shape
    h = _had(x.device)
    codes = torch.empty((rows, width), dtype=torch.float64, device=x.device)
    scales = torch.empty((rows, 1), dtype=torch.float64, device=x.device)
    qmax = 127.0 if bits == 8 else 7.0
    step = max(1, (1 << 26) // width)
    for r in range(0, rows, step):
        v = (x[r:r + step].double().view(-1, 256) @ h.t()).view(-1, width)
        sc = (v.abs().amax(1, keepdim=True) / 16).clamp_min(1e-30) / qmax
        codes[r:r + step] = (v / (16 * sc)).round().clamp(-qmax, qmax)
        scales[r:r + step] = sc
    return codes, scales


def _bf(x):
    return x.to(torch.bfloat16).double()


def _lin(a, w, bits=4):
    (ac, asc), (wc, wsc) = a, _quant(w, bits)
    return (ac @ wc.t()) * asc * wsc.t()


def _silu(g):
    return g / (1 + torch.exp(-g))


def _norm(x, nw):
    x = x.double()
    return _bf(x / torch.sqrt((x * x).mean(1, keepdim=True) + 1e-6) * (nw.double() + 1))


def exact(case, seed):
    r = _raw(case, seed)
    kind = case["kind"]
    if kind == "linear":
        bits = 8 if case["form"] == "int8" else 4
        y = _lin(_quant(r["x"], bits), r["w"], bits)
        return y if r["res"] is None else _bf(y) + r["res"].double()
    if kind == "mlp":
        a = _quant(_norm(r["x"], r["nw"]) if case["norm"] else r["x"])
        g, u = _bf(_lin(a, r["gate"])), _bf(_lin(a, r["up"]))
        return _bf(_lin(_quant(_bf(_bf(_silu(g)) * u)), r["down"])) + r["x"].double()
    if kind == "attention":
        b = case["bits"]
        a = _quant(_norm(r["x"], r["nw"]), b)
        q, k, v = (_lin(a, r[n], b) for n in ("q", "k", "v"))
        m, w = r["att"].shape
        gate = _bf(1 / (1 + torch.exp(-_bf(q).view(m, w // 256, 2, 256)[:, :, 1].reshape(m, w))))
        o = _lin(_quant(_bf(r["att"].double() * gate), b), r["o"], b)
        return q, k, v, _bf(o) + r["x"].double()
    if kind == "moe":
        t, d, f, topk = case["t"], case["d"], case["f"], case["topk"]
        x = r["x"]
        logits = r["logits"].double() if r["logits"] is not None else _bf(x.double() @ r["router"].double().t())
        top, ids = torch.sort(logits, dim=1, descending=True, stable=True)
        top, ids = top[:, :topk], ids[:, :topk]
        p = torch.exp(top - top[:, :1])
        p = _bf(p / p.sum(1, keepdim=True))
        xc, xs = _quant(x)
        out = torch.zeros((t, d), dtype=torch.float64, device=x.device)
        for e in range(EXPERTS):
            tok, rank = (ids == e).nonzero(as_tuple=True)
            for c in range(0, tok.numel(), 16384):
                tk, rk = tok[c:c + 16384], rank[c:c + 16384]
                a = (xc[tk], xs[tk])
                g, u = (_bf(_lin(a, r[n][e * f:(e + 1) * f])) for n in ("gate", "up"))
                y = _bf(_lin(_quant(_bf(_bf(_silu(g)) * u)), r["down"][e * d:(e + 1) * d]))
                out[tk] += _bf(y * p[tk, rk].unsqueeze(1))
        return out
    w = r["w"]
    if case["tiled"]:
        rows, cols = w.shape
        w = w.view(rows // 256, cols // 64, 256, 64).permute(0, 2, 1, 3).reshape(rows, cols)
    scales = _quant(w, case["bits"])[1].view(-1)
    return (None, scales, None) if case["bf6"] else (None, scales)
