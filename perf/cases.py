"""What a user of this library has it do, at the sizes of real use: MoE layers (decode, small batches,
prefill), whole stacks of them, the layer behind its hyper-connection mix, and the dense projections
that share its GEMV.

A case names one operation and its sizes:

  layer   one MoE layer call (`Context.forward`): x [M][H] -> [M][H]
  stack   h <- h + MoE(rmsnorm(h)) through `layers` layers in turn (`Context.residual`)
  hc      the layer behind its hyper-connection mix (`Context.forward_hc`): 4 streams, low rank `lr`
  dense   x [M][k] quantised and projected (`quantize` + `gemv`): -> [M][rows]

H, E, F, k: hidden size, experts, expert width, experts per token.  gate / down: weight formats of the
experts (gate and up share one).  zipf: a router bias that skews the load over the experts.  mass: the
routing takes the fewest experts that reach this share of the top k (0: always k).
"""
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tr-infer_amd"))
import trmoe  # noqa: E402

FMT = {"q4_k": trmoe.FMT_Q4_K, "q6_k": trmoe.FMT_Q6_K, "q8_0": trmoe.FMT_Q8_0, "q5_1": trmoe.FMT_Q5_1,
       "tq4_32": trmoe.FMT_TQ4_32, "tq5_32": trmoe.FMT_TQ5_32, "tq8_32": trmoe.FMT_TQ8_32,
       "tq4_16": trmoe.FMT_TQ4_16, "tq5_16": trmoe.FMT_TQ5_16, "tq8_16": trmoe.FMT_TQ8_16}
# GGUF: bytes of a block and the values that it holds
BLOCK = {"q4_k": (144, 256), "q6_k": (210, 256), "q8_0": (34, 32), "q5_1": (24, 32)}
DEV = "cuda"
HC = 4  # streams of the hyper-connection mix
EPS = 1e-6


# ---- the cases -------------------------------------------------------------------------------------

def _layer(name, M, H=2048, E=512, F=512, k=10, gate="q4_k", down="q4_k", zipf=False, mass=0.0):
    return {"name": name, "op": "layer", "M": M, "H": H, "E": E, "F": F, "k": k, "gate": gate, "down": down,
            "zipf": zipf, "mass": mass}


def _hc(name, M, zipf=False, gate="tq4_32", down="tq5_16", up="tq8_32", H=2560, E=512, F=640, k=10, lr=320):
    return {"name": name, "op": "hc", "M": M, "H": H, "E": E, "F": F, "k": k, "gate": gate, "down": down,
            "zipf": zipf, "mass": 0.0, "lr": lr, "up": up}


def _dense(name, M, rows, cols, fmt, pair=False):
    return {"name": name, "op": "dense", "M": M, "rows": rows, "cols": cols, "fmt": fmt, "pair": pair}


def listed():
    return [
        # decoding one sequence: one token through one layer, two-level activations
        _layer("decode_m1", 1),
        # the same as a serving loop runs it: layer after layer, each with weights of its own
        dict(_layer("stack_m1", 1), op="stack", layers=12),
        # verifying a few drafted tokens
        _layer("verify_m4", 4),
        # decoding sixteen sequences together
        _layer("decode_m16", 16),
        # a short ragged prompt on a smaller model with 8-bit down projections
        _layer("prompt_m37_q8", 37, H=1536, E=128, F=768, k=8, down="q8_0"),
        # prefill, a Zipf-skewed load over the experts
        _layer("prefill_m512", 512, zipf=True),
        # a long prefill: 6-bit down projections, as many experts per token as its routing mass needs
        _layer("prefill_m3072_q6", 3072, down="q6_k", mass=0.9),
        # packed strips, the real shape: the FFN block of one decoded token, mix included
        _hc("hc_decode_m1", 1),
        # and of a prefill, its last rows ragged
        _hc("hc_prefill_m500", 500, zipf=True),
        # the LM head at decode: one token, two-level activations
        _dense("lm_head_m1", 1, 248320, 2560, "tq8_32", pair=True),
        # the smallest projection of a decode step: few rows, long columns
        _dense("low_rank_m1", 1, 320, 10240, "tq8_32", pair=True),
        # an attention projection at prefill
        _dense("dense_m512", 512, 12288, 2560, "tq5_32"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    op = rng.choice(["layer", "layer", "tq", "tq", "dense", "dense", "dense", "stack"])
    if op == "dense":
        fmt = rng.choice(["tq8_32", "tq5_32", "tq4_32", "tq5_16", "q4_k", "q6_k", "q8_0"])
        cols = 256 * _log(rng, 1, 40) if fmt in BLOCK else 32 * _log(rng, 10, 320)
        pair = rng.random() < 0.3
        rows = 16 * _log(rng, 16, 3000)
        M = 1 if pair else _log(rng, 1, 600)
        while rows * cols * M > 16e9:
            M = (M + 1) // 2
        return {"op": "dense", "M": M, "rows": rows, "cols": cols, "fmt": fmt, "pair": pair}
    if op == "tq":
        H, F, E = 256 * rng.randint(4, 10), 16 * rng.randint(10, 40), rng.choice([64, 128, 256, 512])
        c = {"op": rng.choice(["layer", "hc"]), "M": _log(rng, 1, 600), "H": H, "E": E, "F": F, "k": rng.randint(4, 10),
             "gate": rng.choice(["tq4_32", "tq4_32", "tq5_32", "tq8_32"]), "down": rng.choice(["tq5_16", "tq5_16", "tq8_16"]),
             "zipf": rng.random() < 0.5, "mass": 0.0}
        if c["op"] == "hc":
            c.update(lr=32 * rng.randint(2, 10), up="tq8_32")
        return c
    H, F, E = 256 * rng.randint(2, 9), 256 * rng.randint(1, 3), rng.choice([32, 64, 128, 256, 512])
    c = {"op": op, "M": _log(rng, 1, 2500), "H": H, "E": E, "F": F, "k": rng.randint(2, 10), "gate": "q4_k",
         "down": rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_1"]), "zipf": rng.random() < 0.4, "mass": rng.choice([0.0, 0.0, 0.9])}
    if op == "stack":
        c.update(M=_log(rng, 1, 16), layers=rng.randint(2, 8))
    return c


# ---- inputs ----------------------------------------------------------------------------------------

def _matrix_bytes(fmt, rows, k):
    if fmt in BLOCK:
        b, n = BLOCK[fmt]
        return rows * (k // n) * b
    return trmoe.matrix_bytes(FMT[fmt], rows, k)


def _weights(gen, count, rows, k, fmt):
    """`count` quantised matrices [rows][k] as bytes: uniform values, block scales of trained weights' size."""
    if fmt not in BLOCK:
        return trmoe.gen_tq_stack(gen, count, rows, k, FMT[fmt], DEV)
    b, n = BLOCK[fmt]
    t = torch.randint(0, 256, (count, rows * (k // n) * b), dtype=torch.uint8, device=DEV, generator=gen)
    blocks = t.view(-1, b)

    def scale(at, by=1.0):
        v = torch.empty((blocks.shape[0], 1), device=DEV).uniform_(1e-4, 2e-3, generator=gen) * by
        blocks[:, at:at + 2] = v.half().view(torch.uint8)

    if fmt == "q4_k":
        scale(0), scale(2)
    elif fmt == "q6_k":
        scale(208)
    elif fmt == "q8_0":
        scale(0)
    else:
        scale(0), scale(2, -16.0)
    return t


def _moe(gen, c, seed):
    """One layer's tensors."""
    H, E, F = c["H"], c["E"], c["F"]
    w = {"router": torch.randn((E, H), device=DEV, generator=gen) * 0.02,
         "shexp_gate": torch.randn(H, device=DEV, generator=gen) * 0.02,
         "router_bias": torch.from_numpy(trmoe.zipf_bias(seed, E)).to(DEV) if c["zipf"] else None}
    for name, rows, k, fmt in (("gate", F, H, c["gate"]), ("up", F, H, c["gate"]), ("down", H, F, c["down"])):
        w[name] = _weights(gen, E, rows, k, fmt)
        w["sh_" + name] = _weights(gen, 1, rows, k, fmt)[0]
    return w


def _inputs(c, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)

    def normal(*shape):
        return torch.randn(shape, device=DEV, generator=gen)

    if c["op"] == "dense":
        return {"w": _weights(gen, 1, c["rows"], c["cols"], c["fmt"]), "x": normal(c["M"], c["cols"])}
    d = {"layers": [_moe(gen, c, seed + i) for i in range(c.get("layers", 1))]}
    if c["op"] == "stack":
        d["rms"] = [torch.rand(c["H"], device=DEV, generator=gen) * 0.2 + 0.9 for _ in d["layers"]]
        d["h"] = normal(c["M"], c["H"])
    elif c["op"] == "hc":
        d["up"] = _weights(gen, 1, HC * c["H"], c["lr"], c["up"])[0]
        d["xn"], d["lo"] = normal(c["M"], HC, c["H"]), normal(c["M"], c["lr"])
    else:
        d["x"] = normal(c["M"], c["H"])
    return d


def prepare(case, seed):
    c, d = case, _inputs(case, seed)
    if c["op"] == "dense":
        d["y"] = torch.empty((c["M"], c["rows"]), dtype=torch.float32, device=DEV)
        return {"case": c, "in": d}
    lw = [trmoe.LayerWeights(c["H"], c["E"], c["F"], gate_fmt=FMT[c["gate"]], down_fmt=FMT[c["down"]], **w)
          for w in d["layers"]]
    ctx = trmoe.Context(c["H"], c["E"], c["F"], c["k"], c["M"])
    if c["mass"]:
        ctx.set_moe((1, c["k"], c["mass"], trmoe.BASIS_TOP))
    d["out"] = torch.empty((c["M"], c["H"]), dtype=torch.float32, device=DEV)
    return {"case": c, "in": d, "weights": lw, "ctx": ctx}


def run(state):
    c, d = state["case"], state["in"]
    if c["op"] == "dense":
        kb = 16 if c["fmt"] in ("q6_k", "tq5_16") else 32
        q, s, su = trmoe.quantize(d["x"], kb, pair=c["pair"])
        return trmoe.gemv(d["w"], c["rows"], c["cols"], FMT[c["fmt"]], 0, 1, kb, q, s, su, pair=c["pair"], y=d["y"])
    ctx, lw = state["ctx"], state["weights"]
    if c["op"] == "stack":
        h = d["out"].copy_(d["h"])
        for w, r in zip(lw, d["rms"]):
            ctx.residual(w, r, EPS, h)
        return h
    if c["op"] == "hc":
        ctx.forward_hc(lw[0], (d["up"], FMT[c["up"]]), HC, c["lr"], d["xn"], d["lo"], d["out"])
    else:
        ctx.forward(lw[0], d["x"], d["out"])
    return d["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------

def _touched(c):
    """Experts that M tokens are expected to reach, and (token, expert) pairs."""
    E, M, k = c["E"], c["M"], c["k"]
    if c["mass"]:
        k *= 0.9  # near the mean that this routing takes of the top k
    share = [(j + 1) ** -1.1 if c["zipf"] else 1.0 for j in range(E)]  # the draw that the bias is fitted to
    one = [min(1.0, k * p / sum(share)) for p in share]
    return sum(1 - (1 - p) ** M for p in one), k * M


def work(case):
    c = case
    if c["op"] == "dense":
        m = 2 if c["pair"] else c["M"]
        return {"bytes": _matrix_bytes(c["fmt"], c["rows"], c["cols"]) + 4 * c["M"] * (c["cols"] + c["rows"]),
                "flops": 2 * m * c["rows"] * c["cols"]}
    H, E, F, M, n = c["H"], c["E"], c["F"], c["M"], c.get("layers", 1)
    touched, pairs = _touched(c)
    expert = 2 * _matrix_bytes(c["gate"], F, H) + _matrix_bytes(c["down"], H, F)
    b = (touched + 1) * expert + 4 * E * H + 4 * H + 8 * M * H
    f = (2 if M == 1 else 1) * (pairs + M) * 6 * H * F + 2 * M * E * H
    if c["op"] == "hc":
        b += _matrix_bytes(c["up"], HC * H, c["lr"]) + 4 * M * (HC * H + c["lr"]) - 4 * M * H
        f += 2 * M * HC * H * c["lr"]
    return {"bytes": int(n * b), "flops": int(n * f)}


def tolerance(case):
    # 32-bit sums agree with 64-bit ones to 2e-6 as long as every activation rounds to the same int8
    # value.  A few fall on the other side of a tie: 3e-5 of a projection's result at 512 rows, 2e-4 of
    # an MoE layer's (its second quantisation adds flips of its own).
    return {"rel": 2e-4 if case["op"] == "dense" else 1e-3}


# ---- the same in 64 bits ---------------------------------------------------------------------------

def _f16(t):
    """Pairs of bytes [..., 2] as halves, in 32 bits."""
    return t.contiguous().view(torch.float16).float().squeeze(-1)


def _half(t):
    return t.half().double()


def _dequant(raw, rows, k, fmt):
    """The matrix [rows][k] that the bytes hold, in 64 bits."""
    if fmt in BLOCK:
        b = raw.view(rows * (k // BLOCK[fmt][1]), BLOCK[fmt][0])
    if fmt == "q4_k":
        d, dmin, s = _f16(b[:, 0:2]), _f16(b[:, 2:4]), b[:, 4:16].int()
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        return (q.double() * _half(d[:, None] * sc)[..., None] + _half(-(dmin[:, None] * mn))[..., None]).view(rows, k)
    if fmt == "q6_k":
        ql, qh = b[:, 0:128].view(-1, 2, 1, 64), b[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2).view(-1, 2, 4, 32)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).view(-1, 16, 16)
        dd = (_f16(b[:, 208:210])[:, None] * b[:, 192:208].contiguous().view(torch.int8)).half()
        return (q.double() * dd.double()[..., None] + _half(-32.0 * dd.float())[..., None]).view(rows, k)
    if fmt == "q8_0":
        d = _f16(b[:, 0:2])
        q = b[:, 2:].contiguous().view(torch.int8).double() + 128
        return (q * d.double()[:, None] + _half(-128.0 * d)[:, None]).view(rows, k)
    if fmt == "q5_1":
        d, m, qs = _f16(b[:, 0:2]).double(), _f16(b[:, 2:4]).double(), b[:, 8:]
        fifth = (b[:, 4:8, None] >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1
        q = torch.cat([qs & 15, qs >> 4], 1) | (fifth.view(-1, 32) << 4)
        return (q.double() * d[:, None] + m[:, None]).view(rows, k)
    bits, kb = FMT[fmt] >> 8, FMT[fmt] & 255
    strips, nb = (rows + 15) // 16, k // kb
    b = raw.view(strips * nb, -1)
    d, m = (_f16(b[:, o:o + 32].reshape(-1, 16, 2)).double() for o in (0, 32))
    n = kb // 4 if bits == 8 else kb // 8  # chunks of 16 rows by 4 values
    ch = b[:, 64:64 + 64 * n].view(-1, n, 16, 4)
    if bits != 8:
        ch = torch.stack([ch & 15, ch >> 4], 1)
        if bits == 5:
            plane = b[:, 64 + 64 * n:].view(-1, n, 2, 8, 1)
            one = (plane >> torch.arange(8, device=b.device, dtype=torch.uint8)) & 1
            ch = ch | (one.view(-1, n, 2, 16, 4).transpose(1, 2) << 4)
        ch = ch.reshape(-1, 2 * n, 16, 4)
    q = ch.transpose(1, 2).reshape(-1, 16, kb).double()
    w = q * d[..., None] + m[..., None]
    return w.view(strips, nb, 16, kb).transpose(1, 2).reshape(16 * strips, k)[:rows]


def _quant(x, kb):
    """Rows as int8 values times their blocks' scales."""
    v = x.reshape(-1, kb)
    top = v.abs().amax(1, keepdim=True)
    q = torch.round(torch.where(top > 0, v * (127.0 / top), torch.zeros_like(v)))
    return (q * (top / 127.0)).view_as(x)


def _act(x, kb, pair):
    q = _quant(x, kb)
    return q + _quant(x - q, kb) if pair else q


def _exact_layer(c, w, x):
    H, E, F, M, k = c["H"], c["E"], c["F"], c["M"], c["k"]
    pair = M == 1
    logits = x @ w["router"].double().t()
    if w["router_bias"] is not None:
        logits = logits + w["router_bias"].double()
    top, ids = torch.topk(logits, k, dim=1)
    p = torch.softmax(top, 1)
    if c["mass"]:
        before = torch.cumsum(p, 1) - p
        p = torch.where((before < c["mass"]) | (torch.arange(k, device=DEV) < 1), p, torch.zeros_like(p))
        p = p / p.sum(1, keepdim=True)
    share = torch.sigmoid(x @ w["shexp_gate"].double())
    xq = _act(x, 32, pair)

    def expert(rows, by, gate, up, down):
        g = xq[rows] @ _dequant(gate, F, H, c["gate"]).t()
        h = torch.nn.functional.silu(g) * (xq[rows] @ _dequant(up, F, H, c["gate"]).t())
        return (_act(h, 16, pair) * by[:, None]) @ _dequant(down, H, F, c["down"]).t()

    out = expert(torch.arange(M, device=DEV), share, w["sh_gate"], w["sh_up"], w["sh_down"])
    for e in torch.unique(ids[p > 0]).tolist():
        t, slot = torch.nonzero((ids == e) & (p > 0), as_tuple=True)
        out.index_add_(0, t, expert(t, p[t, slot], w["gate"][e], w["up"][e], w["down"][e]))
    return out


def exact(case, seed):
    c, d = case, _inputs(case, seed)
    if c["op"] == "dense":
        xq = _act(d["x"].double(), 16 if c["fmt"] in ("q6_k", "tq5_16") else 32, c["pair"])
        raw, step = d["w"].view(-1), 16 * 512
        per = raw.numel() // (c["rows"] // 16)
        return torch.cat([xq @ _dequant(raw[r // 16 * per:min(r + step, c["rows"]) // 16 * per], min(step, c["rows"] - r),
                                        c["cols"], c["fmt"]).t() for r in range(0, c["rows"], step)], 1)
    if c["op"] == "stack":
        h = d["h"].double()
        for w, r in zip(d["layers"], d["rms"]):
            h = h + _exact_layer(c, w, h * torch.rsqrt(h.square().mean(1, keepdim=True) + EPS) * r.double())
        return h
    if c["op"] == "hc":
        lo = _act(torch.nn.functional.silu(d["lo"].double() / HC), 32, c["M"] == 1)
        gate = torch.sigmoid(lo @ _dequant(d["up"], HC * c["H"], c["lr"], c["up"]).t()).view(c["M"], HC, c["H"])
        return _exact_layer(c, d["layers"][0], (d["xn"].double() * gate).mean(1))
    return _exact_layer(c, d["layers"][0], d["x"].double())
