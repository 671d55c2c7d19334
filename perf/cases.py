"""The work that programs on this framework have it do, as cases that can be timed and checked.

A case is one pass through the public entry points of `runit_mac_amd.dispatch`
(or a whole `DecodeModel` call): single projections, whole transformer layers
at one token (decode) and at many rows (speculative verify, prompt chunks),
the decode step of the 0.5B model and its prefill.  Shapes are those of the
0.5B and 7B Qwen2.5 configurations that bench.py runs; drawn cases take other
sizes of the same ranges, every block format among them.

Weights are N(0, 0.02) quantised per block in the GGUF byte layouts: Q8_0,
Q4_0, Q4_K, Q5_K, Q6_K, in the reference's layouts (q4_0, q4k, q6k) and in
ggml's, which files written by upstream tools hold (q4_0g, q4kg, q5kg, q6kg).
Activations are N(0, 1), or embedding rows.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from runit_mac_amd import dispatch as d
from runit_mac_amd.decode import DecodeConfig, DecodeModel

EPS, THETA = 1e-6, 1e6
HALF = dict(  # 0.5B: 14 query / 2 key-value heads of 64
    hidden=896, heads=14, kv_heads=2, head_dim=64, ff=4864)
SEVEN = dict(  # 7B: 28 / 4 heads of 128
    hidden=3584, heads=28, kv_heads=4, head_dim=128, ff=18944)
VOCAB = 4096  # embedding rows of the layer cases

# (bytes, elements) of a block
BLOCK = {"q8_0": (34, 32), "q4_0": (18, 32), "q4_0g": (18, 32), "q4k": (144, 256),
         "q4kg": (144, 256), "q5kg": (176, 256), "q6k": (210, 256), "q6kg": (210, 256)}
# formats of a model's projections: V and down of a Q4_K_M file are Q6_K
MIX = {"q8_0": dict(a="q8_0", v="q8_0", down="q8_0"),
       "q4_0g": dict(a="q4_0g", v="q4_0g", down="q4_0g"),
       "q4k_m": dict(a="q4k", v="q6k", down="q6k"),
       "q4kg_m": dict(a="q4kg", v="q6kg", down="q6kg"),
       "q5kg_m": dict(a="q5kg", v="q6kg", down="q6kg")}


def listed():
    return [
        # one decode layer of the 0.5B Q8_0 model: launches and their latency
        dict(name="decode_layer_0p5b", kind="layer", mix="q8_0", rows=1, start=511, **HALF),
        # the down projection of a Q4_K_M file (ggml layout) at one token
        dict(name="down_7b", kind="gemv", fmt="q6kg", n=3584, k=18944),
        # one decode layer of a Q4_K_M 7B model with 512 positions of context
        dict(name="decode_layer_7b", kind="layer", mix="q4k_m", rows=1, start=511, **SEVEN),
        # the LM head of that model, its norm fused in (every generated token)
        dict(name="lm_head_7b", kind="head", fmt="q6k", n=152064, k=3584),
        # a gate projection over the rows of a short draft
        dict(name="verify_gemm_7b", kind="gemm", fmt="q4k", rows=8, n=18944, k=3584),
        # a down projection over an odd number of sequences, ggml layout
        dict(name="batch_gemm_7b", kind="gemm", fmt="q6kg", rows=37, n=3584, k=18944),
        # a gate projection of a 512-token prompt, Q8_0 model
        dict(name="prompt_gemm_7b", kind="gemm", fmt="q8_0", rows=512, n=18944, k=3584),
        # one layer of the verification of 7 drafts after 511 positions
        dict(name="verify_layer_7b", kind="layer", mix="q4k_m", rows=8, start=511, **SEVEN),
        # one layer of a 128-token prompt, a Q4_K_M file's ggml layouts
        dict(name="prompt_layer_7b", kind="layer", mix="q4kg_m", rows=128, start=0, **SEVEN),
        # one layer of the last 512-token chunk of a 2048-token prompt
        dict(name="chunk_layer_7b", kind="layer", mix="q4k_m", rows=512, start=1536, **SEVEN),
        # the whole decode step of the 0.5B Q8_0 model, captured once
        dict(name="decode_step_0p5b", kind="step", pos=511),
        # the whole prefill of a 300-token prompt on that model
        dict(name="prefill_0p5b", kind="prefill", rows=300),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("gemv", "gemm", "gemm", "layer", "layer", "layer"))
    if kind == "layer":
        # decode, verify and prompt rows, over models from 0.5B to 7B
        hd = rng.choice((64, 128))
        kv = rng.choice((2, 4))
        group = rng.randint(2, 7)
        rows = rng.choice((1, _log(rng, 2, 512), _log(rng, 2, 512)))
        mix = rng.choice(("q8_0", "q4k_m") if rows == 1 else tuple(MIX))
        if kv * hd == 128 and group % 2:
            group -= 1  # (K-quant blocks hold 256 elements)
        heads = kv * group
        hidden = heads * hd
        if mix == "q8_0" and rng.random() < 0.5:
            hidden, heads, kv, hd = 896, 14, 2, 64  # 28 blocks
        ff = 256 * rng.randint(hidden // 128, hidden // 49 + 1)
        return dict(kind="layer", mix=mix, rows=rows, start=rng.choice((0, _log(rng, 1, 2000))),
                    hidden=hidden, heads=heads, kv_heads=kv, head_dim=hd, ff=ff)
    fmt = rng.choice(tuple(BLOCK))
    el = BLOCK[fmt][1]
    k = el * _log(rng, max(1, 512 // el), 18944 // el)
    most = min(19000, 18944 * 3584 // k)  # weight rows: odd numbers too
    if kind == "gemv":
        # from twice the 0.5B model's largest projection on
        return dict(kind="gemv", fmt=fmt, n=_log(rng, min(most, 8_000_000 // k), most), k=k)
    n = _log(rng, 128, most)
    return dict(kind="gemm", fmt=fmt, rows=_log(rng, 2, 512), n=n, k=k)


# ───────────────────────────── inputs ─────────────────────────────

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda") * std + mean


def _u8(t):
    return t.contiguous().view(torch.uint8)


def _quantise(fmt, w):
    """Blocks [nb, bytes] of w [nb, elements], and the values they stand for (f64)."""
    nb = w.shape[0]
    f16 = torch.float16
    if fmt in ("q8_0", "q4_0", "q4_0g"):
        top = 127 if fmt == "q8_0" else 7
        dq = (w.abs().amax(1, keepdim=True) / top).to(f16)
        q = torch.round(w / dq.float().clamp_min(1e-20)).clamp(-top, top)
        val = lambda: q.double() * dq.double()
        if fmt == "q8_0":
            return torch.cat([_u8(dq), _u8(q.to(torch.int8))], 1), val
        c = (q + 8).to(torch.uint8)
        # the reference's byte i holds elements 2i and 2i + 1, ggml's i and i + 16
        lo, hi = (c[:, 0::2], c[:, 1::2]) if fmt == "q4_0" else (c[:, :16], c[:, 16:])
        return torch.cat([_u8(dq), lo | hi << 4], 1), val
    if fmt in ("q6k", "q6kg"):
        per = 16 if fmt == "q6kg" else 32  # elements of one scale
        s = w.view(nb, 256 // per, per)
        sub = s.abs().amax(2) / 31
        dq = (sub.amax(1, keepdim=True) / 127).to(f16)
        df = dq.float().clamp_min(1e-20)
        sc = torch.round(sub / df).clamp(1, 127)
        q = torch.round(s / (df * sc)[..., None]).clamp(-32, 31)
        val = lambda: ((dq.double() * sc.double())[..., None] * q.double()).view(nb, 256)
        c = (q + 32).to(torch.uint8).view(nb, 2, 4, 32)  # [half][t][l]
        ql = torch.cat([c[:, :, 0:2] & 15 | (c[:, :, 2:4] & 15) << 4], 2)  # [half][t & 1][l]
        qh = (c[:, :, 0] >> 4) | (c[:, :, 1] >> 4) << 2 | (c[:, :, 2] >> 4) << 4 | (c[:, :, 3] >> 4) << 6
        # (the reference reads the even scale slots only)
        sc16 = sc if per == 16 else sc.repeat_interleave(2, 1)
        return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), _u8(sc16.to(torch.int8)),
                          _u8(dq)], 1), val
    # Q4_K / Q5_K: record 2j + hi holds 32 elements; its scale is slot 2j + hi
    # in ggml's layout, j + 4·hi in the reference's
    top = 31 if fmt == "q5kg" else 15
    s = w.view(nb, 8, 32)
    mn = (-s.amin(2)).clamp_min(0)
    sub = (s.amax(2) + mn) / top
    dq = (sub.amax(1, keepdim=True) / 63).to(f16)
    dm = (mn.amax(1, keepdim=True) / 63).to(f16)
    df, dmf = dq.float().clamp_min(1e-20), dm.float().clamp_min(1e-20)
    sc = torch.round(sub / df).clamp(1, 63)
    m = torch.round(mn / dmf).clamp(0, 63)
    q = torch.round((s + (dmf * m)[..., None]) / (df * sc)[..., None]).clamp(0, top)
    val = lambda: ((dq.double() * sc.double())[..., None] * q.double() -
                   (dm.double() * m.double())[..., None]).view(nb, 256)
    slot = list(range(8)) if fmt != "q4k" else [0, 2, 4, 6, 1, 3, 5, 7]  # record of each slot
    S, Mn = sc.to(torch.uint8)[:, slot], m.to(torch.uint8)[:, slot]
    packed = torch.cat([S[:, :4] | (S[:, 4:] >> 4) << 6, Mn[:, :4] | (Mn[:, 4:] >> 4) << 6,
                        S[:, 4:] & 15 | (Mn[:, 4:] & 15) << 4], 1)
    c = q.to(torch.uint8)
    qs = (c[:, 0::2] & 15 | (c[:, 1::2] & 15) << 4).reshape(nb, 128)
    parts = [_u8(dq), _u8(dm), packed]
    if fmt == "q5kg":  # the fifth bit of record r, element l: bit r of byte l
        qh = torch.zeros(nb, 32, dtype=torch.uint8, device=w.device)
        for r in range(8):
            qh |= (c[:, r] >> 4) << r
        parts.append(qh)
    return torch.cat(parts + [qs], 1), val


def _weights(g, fmt, n, k, std=0.02, exact=False):
    """n rows of k weights as the bytes of `fmt`, or as the f64 matrix they stand for."""
    by, el = BLOCK[fmt]
    nb, out, vals = n * k // el, [], []
    step = (1 << 24) // el
    for at in range(0, nb, step):
        b, val = _quantise(fmt, _normal(g, min(step, nb - at), el, std=std))
        if exact:
            vals.append(val())
        else:
            out.append(b)
    if exact:
        return torch.cat(vals).view(n, k)
    return torch.cat(out).reshape(-1)


_ctx = None


def _context():
    """The one context of a program (a stream and a workspace)."""
    global _ctx
    if _ctx is None:
        _ctx = d.HipContext()
        try:  # (its look-up of optional kernels leaves a HIP error behind, which
            torch.zeros(1, device="cuda")  # torch would report on its next launch)
        except RuntimeError:
            pass
    return _ctx


def _p(t):
    return None if t is None else t.data_ptr()


class _View:
    """A device pointer of the framework's as a tensor (while its owner lives)."""

    def __init__(self, ptr, n, typestr):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr,
                                         "data": (int(ptr), False), "version": 3}


def _view(ptr, n, typestr):
    return torch.as_tensor(_View(ptr, n, typestr), device="cuda")


def _layer_inputs(c, seed, exact=False):
    g = _gen(seed)
    f, h, qd, kvd = MIX[c["mix"]], c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    W = lambda fmt, n, k: _weights(g, fmt, n, k, exact=exact)
    s = dict(table=W("q8_0", VOCAB, h), wq=W(f["a"], qd, h), wk=W(f["a"], kvd, h),
             wv=W(f["v"], kvd, h), wo=W(f["a"], h, qd), wg=W(f["a"], c["ff"], h),
             wu=W(f["a"], c["ff"], h), wd=W(f["down"], h, c["ff"]))
    for b, n in (("bq", qd), ("bk", kvd), ("bv", kvd)):
        s[b] = _normal(g, n, std=0.02).half()
    s["norm1"], s["norm2"] = _normal(g, h, std=0.02, mean=1.0), _normal(g, h, std=0.02, mean=1.0)
    span = c["start"] + c["rows"]
    s["kc"], s["vc"] = (_normal(g, c["kv_heads"], span, c["head_dim"]) for _ in range(2))
    s["tok"] = torch.randint(0, VOCAB, (c["rows"],), generator=g, device="cuda", dtype=torch.int32)
    return s


def _step_config(c):
    return DecodeConfig(max_seq=1024)


def _model_inputs(cfg, seed, exact=False):
    """Every tensor of the 0.5B Q8_0 model, by name."""
    g = _gen(seed)
    h, q, kv, ff = cfg.hidden, cfg.q_dim, cfg.kv_dim, cfg.ff
    W = lambda n, k: _weights(g, "q8_0", n, k, exact=exact)
    cache = cfg.kv_heads * cfg.max_seq * cfg.head_dim
    layers = []
    for _ in range(cfg.layers):
        layers.append(dict(
            wq=W(q, h), wk=W(kv, h), wv=W(kv, h), wo=W(h, q), wg=W(ff, h), wu=W(ff, h), wd=W(h, ff),
            bq=_normal(g, q, std=0.02).half(), bk=_normal(g, kv, std=0.02).half(),
            bv=_normal(g, kv, std=0.02).half(), attn_norm=_normal(g, h, std=0.02, mean=1.0),
            ffn_norm=_normal(g, h, std=0.02, mean=1.0), kc=_normal(g, cache), vc=_normal(g, cache)))
    return layers, _normal(g, h, std=0.02, mean=1.0), W(cfg.vocab, h)


def _tokens(seed, n, vocab):
    return np.random.default_rng(seed).integers(0, vocab, n)


def prepare(case, seed):
    ctx, c = _context(), case
    s = dict(case=c, ctx=ctx)
    if c["kind"] in ("step", "prefill"):
        cfg = _step_config(c)
        m = DecodeModel(ctx, cfg, seed=7)
        layers, norm, embd = _model_inputs(cfg, seed)
        for L, t in zip(m.layers, layers):
            for name, v in t.items():
                v = _u8(v).reshape(-1)
                _view(L[name], v.numel(), "|u1").copy_(v)
        _view(m.final_norm, cfg.hidden, "<f4").copy_(norm)
        _view(m.embd, embd.numel(), "|u1").copy_(embd)
        torch.cuda.synchronize()
        s.update(model=m, tokens=_tokens(seed, c.get("rows", 1), cfg.vocab))
        if c["kind"] == "step":
            # results in tensors of the program's own (they outlive the model)
            s["logits"] = torch.zeros(cfg.vocab, device="cuda")
            s["token"] = torch.zeros(1, device="cuda", dtype=torch.int32)
            torch.cuda.synchronize()
            m.logits, m.token = _p(s["logits"]), _p(s["token"])
            m.set_token(int(s["tokens"][0]))
            s["graph"] = m.capture(c["pos"])
        return s
    if c["kind"] == "layer":
        s.update(_layer_inputs(c, seed))
        M, h, qd, kvd = c["rows"], c["hidden"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
        for name, n in (("x", h), ("xm", h), ("xn", h), ("q", qd), ("k", kvd), ("v", kvd),
                        ("att", qd), ("g", c["ff"]), ("u", c["ff"])):
            s[name] = torch.empty(M, n, device="cuda")
    else:
        g = _gen(seed)
        s["w"] = _weights(g, c["fmt"], c["n"], c["k"])
        rows = c.get("rows", 1)
        s["x"] = _normal(g, rows, c["k"])
        if c["kind"] == "gemv":
            s["res"] = _normal(g, c["n"])
        if c["kind"] == "head":
            s["norm"] = _normal(g, c["k"], std=0.02, mean=1.0)
        s["y"] = torch.empty(rows, c["n"], device="cuda")
    torch.cuda.synchronize()  # the framework has a stream of its own
    return s


# ───────────────────────────── one pass ─────────────────────────────

def _run_layer(s):
    c, ctx = s["case"], s["ctx"]
    f, M, h, ff, start = MIX[c["mix"]], c["rows"], c["hidden"], c["ff"], c["start"]
    hd, nh, nkv = c["head_dim"], c["heads"], c["kv_heads"]
    qd, kvd, span = nh * hd, nkv * hd, start + M
    P = {k: _p(v) for k, v in s.items() if isinstance(v, torch.Tensor)}
    if M == 1:  # decode: DecodeModel.step_fused's launches of one layer
        d.embed_q8_0_f32(ctx, P["table"], P["tok"], P["x"], h)
        name = "q8_0" if f["a"] == "q8_0" else "q4k_q6k"
        getattr(d, f"rms_norm_fused_qkv_bias_{name}_f32")(
            ctx, P["wq"], P["wk"], P["wv"], P["x"], P["norm1"], EPS, P["q"], P["k"], P["v"],
            P["bq"], P["bk"], P["bv"], qd, kvd, h)
        getattr(d, f"decode_attention_rope_oproj_{f['a']}_f32")(
            ctx, P["q"], P["k"], P["v"], P["kc"], P["vc"], P["wo"], P["x"], start, span, nh, nkv,
            hd, THETA, h)
        getattr(d, f"rms_norm_fused_ffn_{f['a']}_f32")(ctx, P["wg"], P["wu"], P["x"], P["norm2"],
                                                       EPS, P["g"], ff, h)
        getattr(d, f"gemv_{f['down']}_add_f32_f32in")(ctx, P["wd"], P["g"], P["x"], P["x"], h, ff)
    else:  # verify / prompt rows: DecodeModel.verify_pass's calls of one layer
        d.embed_rows_f32(ctx, "q8_0", P["table"], P["tok"], P["x"], h, M)
        d.gemm_qkv_rope_f32(ctx, (f["a"], f["a"], f["v"]), P["wq"], P["wk"], P["wv"], P["bq"],
                            P["bk"], P["bv"], P["x"], P["norm1"], EPS, P["xn"], P["q"], P["k"],
                            P["v"], P["kc"], P["vc"], M, h, qd, kvd, hd, start, THETA, span)
        d.gemm_attn_ffn_block_f32(ctx, P["q"], P["kc"], P["vc"], span, nh, nkv, hd, span, start,
                                  P["att"], (f["a"], f["a"], f["a"], f["down"]), P["wo"], P["wg"],
                                  P["wu"], P["wd"], P["x"], P["xm"], P["norm2"], EPS, P["g"],
                                  P["u"], P["xn"], M, h, ff)
    return {"x": s["x"], "k": s["kc"][:, start:], "v": s["vc"][:, start:]}


def run(state):
    s = state
    c, ctx = s["case"], s["ctx"]
    kind = c["kind"]
    if kind == "layer":
        return _run_layer(s)
    if kind == "gemv":
        getattr(d, f"gemv_{c['fmt']}_add_f32_f32in")(ctx, _p(s["w"]), _p(s["x"]), _p(s["y"]),
                                                     _p(s["res"]), c["n"], c["k"])
    elif kind == "head":
        getattr(d, f"rms_norm_gemv_{c['fmt']}_f32in_f32out")(
            ctx, _p(s["w"]), _p(s["x"]), _p(s["norm"]), EPS, _p(s["y"]), c["n"], c["k"])
    elif kind == "gemm":
        getattr(d, f"gemm_{c['fmt']}_f32")(ctx, _p(s["w"]), _p(s["x"]), _p(s["y"]), c["rows"],
                                           c["n"], c["k"])
    elif kind == "step":
        s["model"].set_token(int(s["tokens"][0]))  # as a program that samples on the host does
        s["graph"].launch()
        return {"logits": s["logits"], "token": s["token"]}
    else:
        return {"logits": s["model"].prefill(s["tokens"])}
    return s["y"]


# ───────────────────────────── cost and bounds ─────────────────────────────

def _matrix(fmt, n, k):
    by, el = BLOCK[fmt]
    return n * k // el * by


def _layer_work(M, start, h, qd, kvd, ff, nh, nkv, hd, f):
    mats = ((f["a"], qd, h), (f["a"], kvd, h), (f["v"], kvd, h), (f["a"], h, qd), (f["a"], ff, h),
            (f["a"], ff, h), (f["down"], h, ff))
    pairs = sum(start + r + 1 for r in range(M))
    return (sum(_matrix(*m) for m in mats) + 8 * nkv * hd * (start + 2 * M) + 8 * M * h,
            2 * M * sum(n * k for _, n, k in mats) + 4 * pairs * nh * hd)


def work(case):
    c = case
    if c["kind"] == "layer":
        hd = c["head_dim"]
        b, f = _layer_work(c["rows"], c["start"], c["hidden"], c["heads"] * hd, c["kv_heads"] * hd,
                           c["ff"], c["heads"], c["kv_heads"], hd, MIX[c["mix"]])
        return {"bytes": b, "flops": f}
    if c["kind"] in ("step", "prefill"):
        g = _step_config(c)
        M, start = (1, c["pos"]) if c["kind"] == "step" else (c["rows"], 0)
        b, f = _layer_work(M, start, g.hidden, g.q_dim, g.kv_dim, g.ff, g.heads, g.kv_heads,
                           g.head_dim, MIX["q8_0"])
        return {"bytes": g.layers * b + _matrix("q8_0", g.vocab, g.hidden) + 4 * g.vocab,
                "flops": g.layers * f + 2 * g.vocab * g.hidden}
    M, n, k = c.get("rows", 1), c["n"], c["k"]
    extra = 4 * n if c["kind"] == "gemv" else 4 * k if c["kind"] == "head" else 0
    return {"bytes": _matrix(c["fmt"], n, k) + 4 * M * (n + k) + extra, "flops": 2 * M * n * k}


def tolerance(case):
    # about four times the error against 64 bits measured on these cases
    if case["kind"] in ("step", "prefill"):
        return {"rel": 4e-5, "max": 1e-3}  # 24 layers, one after the other, in 32 bits
    if case["kind"] == "layer":
        # RoPE angles of up to some thousand radians in 32 bits, then softmax
        # and four projections (2e-5 at position 2047, 1e-6 at the first ones)
        return {"rel": 8e-5, "max": 2e-3}
    return {"rel": 2e-6, "max": 4e-5}  # one sum in 32 bits


# ───────────────────────────── the same in 64 bits ─────────────────────────────

def _norm64(x, gamma):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * gamma.double()


def _rope64(t, start):  # [rows][heads][dim], pairs (i, i + dim / 2)
    rows, _, hd = t.shape
    half = hd // 2
    i = torch.arange(half, device=t.device, dtype=torch.float64)
    pos = torch.arange(start, start + rows, device=t.device, dtype=torch.float64)
    a = (pos[:, None] / THETA ** (2 * i / hd))[:, None, :]
    lo, hi = t[..., :half], t[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _layer64(x, s, start, nh, nkv, hd):
    """One layer of x [rows][hidden]; the caches [heads][positions][dim] are written."""
    M = x.shape[0]
    xn = _norm64(x, s["norm1"])
    q, k, v = (xn @ s[w].T + s[b].double() for w, b in (("wq", "bq"), ("wk", "bk"), ("wv", "bv")))
    kc, vc = s["kc"], s["vc"]
    kc[:, start:start + M] = _rope64(k.view(M, nkv, hd), start).transpose(0, 1)
    vc[:, start:start + M] = v.view(M, nkv, hd).transpose(0, 1)
    q = _rope64(q.view(M, nh, hd), start)
    span, out = start + M, torch.empty(M, nh, hd, dtype=torch.float64, device=x.device)
    seen = torch.arange(span, device=x.device)[None, :] <= start + torch.arange(M, device=x.device)[:, None]
    for i in range(nh):
        g = i // (nh // nkv)
        p = (q[:, i] @ kc[g, :span].T / math.sqrt(hd)).masked_fill(~seen, -math.inf).softmax(-1)
        out[:, i] = p @ vc[g, :span]
    x = x + out.view(M, nh * hd) @ s["wo"].T
    xn = _norm64(x, s["norm2"])
    gate = xn @ s["wg"].T
    return x + (gate / (1 + torch.exp(-gate)) * (xn @ s["wu"].T)) @ s["wd"].T


def exact(case, seed):
    c = case
    if c["kind"] == "layer":
        s = _layer_inputs(c, seed, exact=True)
        s["kc"], s["vc"] = s["kc"].double(), s["vc"].double()
        x = _layer64(s["table"][s["tok"].long()], s, c["start"], c["heads"], c["kv_heads"], c["head_dim"])
        return {"x": x, "k": s["kc"][:, c["start"]:].clone(), "v": s["vc"][:, c["start"]:].clone()}
    if c["kind"] in ("step", "prefill"):
        cfg = _step_config(c)
        M, start = (1, c["pos"]) if c["kind"] == "step" else (c["rows"], 0)
        layers, norm, embd = _model_inputs(cfg, seed, exact=True)
        x = embd[torch.from_numpy(_tokens(seed, M, cfg.vocab)).cuda()]
        for L in layers:
            L["norm1"], L["norm2"] = L["attn_norm"], L["ffn_norm"]
            for n in ("kc", "vc"):
                L[n] = L[n].double().view(cfg.kv_heads, cfg.max_seq, cfg.head_dim)
            x = _layer64(x, L, start, cfg.heads, cfg.kv_heads, cfg.head_dim)
        y = _norm64(x[-1], norm) @ embd.T
        return {"logits": y, "token": None} if c["kind"] == "step" else {"logits": y}
    g = _gen(seed)
    w = _weights(g, c["fmt"], c["n"], c["k"], exact=True)
    x = _normal(g, c.get("rows", 1), c["k"]).double()
    if c["kind"] == "gemv":
        return x @ w.T + _normal(g, c["n"]).double()
    if c["kind"] == "head":
        x = _norm64(x, _normal(g, c["k"], std=0.02, mean=1.0))
    return x @ w.T
