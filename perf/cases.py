"""Timed cases of the W8A8 linear and the fused DiT kernels.

Each case is one thing a program on this library has it do, called through
h3mi's public functions: a W8A8 linear (per-token or ConvRot quantizer, then
the GEMM), a fused norm / gate, the q/k norm with rotary embedding, or the MLP
half of a DiT block built from them.  Token counts run from one row (a
conditioning vector) over prompts (tens to hundreds of rows) and per-GPU
shares of a clip (a few thousand) to whole clips (19200, 32768 or 38400 rows);
widths are those of the hidden-5120 block (40 heads x 128, MLP 13824), of the
hidden-5376 H3 layers (56 heads x 128, fc1 28672, fc2 14336), of the single
3072-wide linear, or generic multiples that the entry points accept.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "minimax-h3-multi-dgx-spark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import h3mi  # noqa: E402

EPS = 1e-6
BF16 = torch.bfloat16

# The largest listed linear: no drawn case multiplies more.
_MAX_MKN = 32768 * 5120 * 15360


def listed():
    return [
        # A short prompt's cross-attention K/V projection: few rows against a whole weight; latency counts.
        {"name": "linear_kv_37", "kind": "linear", "m": 37, "k": 5120, "n": 10240, "bias": True},
        # The same projection for the 512 text tokens of a block.
        {"name": "linear_kv_512", "kind": "linear", "m": 512, "k": 5120, "n": 10240, "bias": True},
        # A single mid-sized linear.
        {"name": "linear_3072", "kind": "linear", "m": 2048, "k": 3072, "n": 3072, "bias": True},
        # The fused QKV projection of a whole clip: the largest product.
        {"name": "linear_qkv_32768", "kind": "linear", "m": 32768, "k": 5120, "n": 15360, "bias": True},
        # H3's attention output projection (ConvRot checkpoint) on an uneven per-GPU share of the tokens.
        {"name": "convrot_out_4799", "kind": "convrot", "m": 4799, "k": 7168, "n": 5376, "act": "none"},
        # H3's second MLP linear for a 19200-token clip: SwiGLU and rotation in the quantizer.
        {"name": "convrot_fc2_19200", "kind": "convrot", "m": 19200, "k": 14336, "n": 5376, "act": "swiglu"},
        # The first norm of a block for the text tokens: a small, launch-bound call.
        {"name": "norm_mod_512", "kind": "norm", "op": "norm_mod", "s": 512, "n": 5120, "r": 1},
        # Norm with the next linear's quantizer fused, an odd share of a clip whose rows use two modulation rows.
        {"name": "norm_mod_q_2401", "kind": "norm", "op": "norm_mod_q", "s": 2401, "n": 5376, "r": 2},
        # The second norm of a block, with the attention's gated residual, for a whole clip.
        {"name": "gate_norm_mod_19200", "kind": "norm", "op": "gate_norm_mod_", "s": 19200, "n": 5376, "r": 1},
        # The MLP's gated residual for a whole clip: the largest elementwise pass.
        {"name": "gate_32768", "kind": "norm", "op": "gate_", "s": 32768, "n": 5120, "r": 1},
        # q/k norm and rotary embedding of a clip, on views of the qkv projection.
        {"name": "rope_19200", "kind": "rope", "s": 19200, "heads": 56, "dim": 128, "rot": 128},
        # The MLP half of an H3 block on an eighth of a clip: gate + norm, fc1, SwiGLU, fc2, gate, each a call.
        {"name": "mlp_half_2400", "kind": "mlp", "m": 2400, "k": 5376, "f": 14336},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["linear", "convrot", "norm", "rope", "mlp"], [4, 2, 4, 1, 1])[0]
    if kind == "linear":
        k, n = rng.choice([(3072, 3072), (5120, 15360), (5120, 13824), (13824, 5120), (5120, 5120), (5120, 10240),
                           (128 * _log(rng, 3, 112), 4 * _log(rng, 18, 5376)),
                           (128 * _log(rng, 3, 112), 4 * _log(rng, 18, 5376))])
        m = _log(rng, 1, min(32768, _MAX_MKN // (k * n)))
        return {"kind": kind, "m": m, "k": k, "n": n, "bias": rng.random() < 0.5}
    if kind == "convrot":
        k, n, act = rng.choice([(5376, 21504, "none"), (7168, 5376, "none"), (5376, 28672, "none"),
                                (14336, 5376, "swiglu"), (256 * _log(rng, 2, 56), 8 * _log(rng, 16, 2688), "none"),
                                (256 * _log(rng, 2, 56), 8 * _log(rng, 16, 2688), "swiglu")])
        return {"kind": kind, "m": _log(rng, 1, min(38400, _MAX_MKN // (k * n))), "k": k, "n": n, "act": act}
    if kind == "norm":
        op = rng.choice(["norm_mod", "gate_norm_mod_", "gate_", "norm_mod_q", "gate_norm_mod_q_"])
        n = rng.choice([5120, 5376, 3072, 8 * rng.randint(16, 1024)])
        s = _log(rng, 1, 38400)
        return {"kind": kind, "op": op, "s": s, "n": n, "r": min(s, rng.choice([1, 1, 2, 5]))}
    if kind == "rope":
        heads, dim = rng.choice([(56, 128), (40, 128), (24, 64), (12, 256)])
        return {"kind": kind, "s": _log(rng, 1, 38400), "heads": heads, "dim": dim, "rot": rng.choice([dim, dim, dim // 2])}
    k, f = rng.choice([(5376, 14336), (3072, 8192)])
    return {"kind": kind, "m": _log(rng, 8, 4800), "k": k, "f": f}


# ------------------------------------------------------------------ inputs


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape, scale=1.0, mean=0.0):
    t = torch.randn(*shape, generator=g, device="cuda")
    return (t * scale + mean).to(BF16)


def _activations(g, m, k):
    """N(0, 1) with 0.1% of the elements 20 times larger, as activations have outlier channels and tokens."""
    x = torch.randn(m, k, generator=g, device="cuda")
    x = torch.where(torch.rand(m, k, generator=g, device="cuda") < 1e-3, x * 20, x)
    return x.to(BF16)


def _weight(g, n, k, unit=False):
    """int8 weight and per-channel scales: U(1e-3, 1e-2), or (unit) such that unit inputs give unit outputs."""
    w = torch.randint(-127, 128, (n, k), generator=g, device="cuda", dtype=torch.int8)
    u = torch.rand(n, generator=g, device="cuda")
    return w, ((0.5 + u) / (73.3 * math.sqrt(k)) if unit else 1e-3 + 9e-3 * u)


def _segments(g, s, r):
    """Row -> modulation row: r runs of tokens in order, as a batch of segments has them."""
    cuts = torch.randint(0, s + 1, (r - 1,), generator=g, device="cuda").sort().values if r > 1 else None
    rows = torch.arange(s, device="cuda")
    return (torch.bucketize(rows, cuts, right=True) if r > 1 else torch.zeros_like(rows)).to(torch.int32)


def _modulation(g, n, r):
    """w, s1 = 1 + scale, shift, gate."""
    w = _normal(g, n, scale=0.02, mean=1.0)
    s1 = 1.0 + _normal(g, r, n, scale=0.1)
    return w, s1.contiguous(), _normal(g, r, n, scale=0.1), _normal(g, r, n, scale=0.1)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    st = {"case": case}
    if kind == "linear":
        st["x"] = _activations(g, case["m"], case["k"])
        st["w"], st["ws"] = _weight(g, case["n"], case["k"])
        st["bias"] = _normal(g, case["n"], scale=0.02) if case["bias"] else None
    elif kind == "convrot":
        wide = 2 if case["act"] == "swiglu" else 1
        st["x"] = _activations(g, case["m"], case["k"] * wide)
        st["w"], st["ws"] = _weight(g, case["n"], case["k"])
    elif kind == "norm":
        s, n, r = case["s"], case["n"], case["r"]
        st["x"] = _normal(g, s, n)
        st["o"] = _normal(g, s, n) if case["op"].startswith("gate") else None
        st["w"], st["s1"], st["sh"], st["g"] = _modulation(g, n, r)
        st["ridx"] = _segments(g, s, r)
    elif kind == "rope":
        s, heads, dim, rot = case["s"], case["heads"], case["dim"], case["rot"]
        st["qkv"] = _normal(g, s, 3 * heads * dim)
        ang = 6.2831853 * torch.rand(s, rot // 2, generator=g, device="cuda")
        rows = torch.stack([ang.cos(), -ang.sin(), ang.sin(), ang.cos()], -1)
        st["tab"] = rows.reshape(1, s, rot // 2, 2, 2).to(BF16)
        st["qw"], st["kw"] = _normal(g, dim, scale=0.02, mean=1.0), _normal(g, dim, scale=0.02, mean=1.0)
        st["q"], st["k"] = (st["qkv"][:, i * heads * dim:(i + 1) * heads * dim].reshape(1, s, heads, dim) for i in (0, 1))
    else:
        m, k, f = case["m"], case["k"], case["f"]
        st["x"], st["o"] = _normal(g, m, k), _normal(g, m, k)
        st["w"], st["s1"], st["sh"], st["g"] = _modulation(g, k, 1)
        st["g2"] = _normal(g, 1, k, scale=0.1)
        st["w1"], st["ws1"] = _weight(g, 2 * f, k, unit=True)
        st["w2"], st["ws2"] = _weight(g, k, f, unit=True)
        st["ridx"] = _segments(g, m, 1)
    return st


# ------------------------------------------------------------------ one pass


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "linear":
        return h3mi.w8a8_linear(st["x"], st["w"], st["ws"], bias=st["bias"])
    if kind == "convrot":
        xq, xs = h3mi.quantize_rowwise_convrot(st["x"], case["act"])
        return h3mi.int8_mm_scaled(xq, st["w"], xs, st["ws"])
    if kind == "norm":
        x, o, g, w, ridx, s1, sh = (st[k] for k in ("x", "o", "g", "w", "ridx", "s1", "sh"))
        op = case["op"]
        if op == "norm_mod":
            return h3mi.norm_mod(x, w, EPS, ridx, s1, sh)
        if op == "gate_norm_mod_":
            return x, h3mi.gate_norm_mod_(x, o, g, w, EPS, ridx, s1, sh)
        if op == "gate_":
            return h3mi.gate_(x, o, g, ridx)
        if op == "norm_mod_q":
            return h3mi.norm_mod_q(x, w, EPS, ridx, s1, sh)
        return x, h3mi.gate_norm_mod_q_(x, o, g, w, EPS, ridx, s1, sh)
    if kind == "rope":
        return h3mi.rms_rope_split_half_(st["q"], st["k"], st["tab"], st["qw"], st["kw"], epsilon=EPS)
    x, ridx = st["x"], st["ridx"]
    h = h3mi.gate_norm_mod_(x, st["o"], st["g"], st["w"], EPS, ridx, st["s1"], st["sh"])
    hq, hs = h3mi.quantize_rowwise_convrot(h)
    a = h3mi.int8_mm_scaled(hq, st["w1"], hs, st["ws1"])
    aq, as_ = h3mi.quantize_rowwise_convrot(a, "swiglu")
    y = h3mi.int8_mm_scaled(aq, st["w2"], as_, st["ws2"])
    return y, h3mi.gate_(x, y, st["g2"], ridx)


# ------------------------------------------------------------------ what a pass cannot do without


def work(case):
    kind = case["kind"]
    if kind in ("linear", "convrot"):
        m, k, n = case["m"], case["k"], case["n"]
        wide = 2 if case.get("act") == "swiglu" else 1
        return {"bytes": 2 * m * k * wide + n * k + 4 * n + (2 * n if case.get("bias") else 0) + 2 * m * n,
                "flops": 2 * m * k * n}
    if kind == "norm":
        s, n, r, op = case["s"], case["n"], case["r"], case["op"]
        per = {"norm_mod": 4, "gate_norm_mod_": 8, "gate_": 6, "norm_mod_q": 3, "gate_norm_mod_q_": 7}[op]
        tables = 2 * n * (r if op == "gate_" else 1 + (3 if op.startswith("gate") else 2) * r)
        return {"bytes": per * s * n + tables + 4 * s + (4 * s if op.endswith(("_q", "_q_")) else 0), "flops": 0}
    if kind == "rope":
        s, hd = case["s"], case["heads"] * case["dim"]
        return {"bytes": 8 * s * hd + 4 * s * case["rot"] + 4 * case["dim"], "flops": 0}
    m, k, f = case["m"], case["k"], case["f"]
    # x and o read, x and the MLP's output written; both weights read
    return {"bytes": 8 * m * k + 3 * k * f + 4 * (2 * f + k) + 10 * k + 4 * m, "flops": 6 * m * k * f}


# ------------------------------------------------------------------ how close two correct results are


def tolerance(case):
    """About four times what the present path shows against exact()."""
    kind = case["kind"]
    if kind in ("linear", "convrot"):
        # one bf16 rounding of an exact integer product, and quantizer ties: 1.7e-3, largest 2.0e-2
        return {"rel": 7e-3, "max": 0.08}
    if kind == "norm":
        if case["op"].endswith(("_q", "_q_")):
            # h's bf16 roundings move 9% of the int8 values by one: 9.1e-3, largest 3.2e-2
            return {"rel": 3.6e-2, "max": 0.13, "differ": 0.36}
        return {"rel": 1.3e-2, "max": 0.06}  # three bf16 roundings: 3.3e-3, largest 1.6e-2
    if kind == "rope":
        return {"rel": 1e-2, "max": 0.06}  # two bf16 roundings: 2.4e-3, largest 1.6e-2
    # two norms' and two linears' roundings through two int8 quantizers: 1.9e-2, largest 0.16
    return {"rel": 7.7e-2, "max": 0.64}


def _quant64(u):
    """(q, s) of rows u in 64 bits; the scale is stored in 32 bits, so q is taken against the stored one."""
    s = (u.abs().amax(1, keepdim=True) / 127).float().double()
    return torch.where(s > 0, torch.round(u / s.clamp_min(1e-300)), torch.zeros_like(u)).clamp_(-127, 127), s


def _rotate64(u):
    h = torch.ones(1, 1, device="cuda", dtype=torch.float64)
    while h.shape[0] < 256:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return (u.reshape(-1, 256) @ (h / 16)).reshape(u.shape)


def _swiglu64(u):
    a, b = u.chunk(2, dim=1)
    return a * torch.sigmoid(a) * b


def _linear64(u, w, ws, bias=None):
    q, s = _quant64(u)
    y = (q @ w.double().t()).mul_(s).mul_(ws.double())
    return y if bias is None else y.add_(bias.double())


def _norm64(x, st):
    y = x * torch.rsqrt(x.square().mean(1, keepdim=True) + EPS) * st["w"].double()
    i = st["ridx"].long()
    return y * st["s1"].double()[i] + st["sh"].double()[i]


def exact(case, seed):
    st, kind = prepare(case, seed), case["kind"]
    if kind == "linear":
        return _linear64(st["x"].double(), st["w"], st["ws"], st["bias"])
    if kind == "convrot":
        x = st["x"].double()
        return _linear64(_rotate64(_swiglu64(x) if case["act"] == "swiglu" else x), st["w"], st["ws"])
    if kind == "norm":
        op, x = case["op"], st["x"].double()
        if op.startswith("gate"):
            x = x + st["o"].double() * st["g"].double()[st["ridx"].long()]
        if op == "gate_":
            return x
        h = _norm64(x, st)
        if op.endswith(("_q", "_q_")):
            q, s = _quant64(h)
            h = (q.to(torch.int8), s)
        return (x, h) if op.startswith("gate") else h
    if kind == "rope":
        out = []
        for t, w in ((st["q"], st["qw"]), (st["k"], st["kw"])):
            y = t.double()
            y = y * torch.rsqrt(y.square().mean(-1, keepdim=True) + EPS) * w.double()
            half = case["rot"] // 2
            r = st["tab"].double().unsqueeze(2)  # [1, s, 1, half, 2, 2]
            a, b = y[..., :half], y[..., half:2 * half]
            out.append(torch.cat([r[..., 0, 0] * a + r[..., 0, 1] * b, r[..., 1, 0] * a + r[..., 1, 1] * b,
                                  y[..., 2 * half:]], -1))
        return tuple(out)
    x = st["x"].double() + st["o"].double() * st["g"].double()[st["ridx"].long()]
    a = _linear64(_rotate64(_norm64(x, st)), st["w1"], st["ws1"])
    y = _linear64(_rotate64(_swiglu64(a)), st["w2"], st["ws2"])
    return y, x + y * st["g2"].double()
