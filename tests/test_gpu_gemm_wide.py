"""The wide batched GEMM (k_gemmw_<fmt>, more than 32 activation rows, fewer
where nothing else tiles K) of every block format against the oracle's per-row
f64 GEMV of the same packed blocks, at the edges of its tiles: rows around one
and two 64-row chunks, weight rows around 256-row tiles, K of one block, of an
odd number of blocks, of one and several super-blocks, and K ranges split over
workgroups.  Tolerance: every output within 1e-4·Σ|w·x| (gpu_helpers); the
form's own error is the 22 bits of the f16 pairs and some ten f32 roundings,
below 1e-6·Σ|w·x|, checked too."""
import os

import numpy as np
import pytest

import oracle_lib as ora
import test_gpu_gemm_set
from runit_mac_amd import dispatch as d
from gpu_helpers import check_close, device_weights
from test_gpu_fused import ffn_check

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    """A context whose calls take the wide form from 33 rows on, however small
    (by default from 1.6e9 rows × weights on, and where no other form fits)."""
    os.environ["RUNIT_GEMM_WIDE_WORK"] = "0"
    try:
        c = d.HipContext()
    finally:
        del os.environ["RUNIT_GEMM_WIDE_WORK"]
    yield c
    c.close()


SMALL = ("q8_0", "q4_0", "q4_0g", "q5_0")
SUPER = ("q4k", "q4kg", "q5k", "q5kg", "q6k", "q6kg")


def _check(ctx, fmt, m, n, k, seed):
    w, raw = device_weights(ctx, fmt, n, k, seed)
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[m // 2] *= 1e-3  # rows of their own scale, and an all-zero one
    x[m - 1] = 0.0
    y = ctx.new_buffer(4 * (m * n + 64))
    y.write(np.full(m * n + 64, 7.0, np.float32))
    getattr(d, f"gemm_{fmt}_f32")(ctx, w, ctx.buffer_from(x), y, m, n, k)
    odd = "_o" if (k // d.BLOCK[fmt][0]) % 2 and fmt not in ("q4k", "q4kg", "q5k", "q5kg") else ""
    assert d.last_launch_name(ctx) in (f"k_gemmw_{fmt}{odd}", "k_gemm_split_sum")
    ctx.flush()
    got = y.read(np.float32, m * n + 64)
    assert np.all(got[m * n:] == 7.0), "past the last row"
    ref, sabs = ora.gemv(fmt, raw, x, n, k)
    check_close(got[:m * n], ref.ravel(), sabs.ravel(), f"{fmt} {m}x{n}x{k}")
    err = np.abs(got[:m * n].astype(np.float64) - ref.ravel())
    assert np.all(err <= 1e-6 * sabs.ravel()), f"{fmt} {m}x{n}x{k}: {(err / np.maximum(sabs.ravel(), 1e-30)).max():.2e}"


@pytest.mark.parametrize("fmt", SMALL)
@pytest.mark.parametrize("m,n,k", [(33, 1, 32), (64, 257, 96), (65, 300, 2080), (130, 511, 896)])
def test_wide_gemm_block_formats(ctx, fmt, m, n, k):
    _check(ctx, fmt, m, n, k, 900 + m)


@pytest.mark.parametrize("fmt", SUPER)
@pytest.mark.parametrize("m,n,k", [(33, 3, 256), (64, 257, 768), (129, 300, 4096)])
def test_wide_gemm_super_block_formats(ctx, fmt, m, n, k):
    _check(ctx, fmt, m, n, k, 920 + m)


@pytest.mark.parametrize("fmt,m,n,k", [("q4_0", 5, 70, 32), ("q4_0g", 8, 257, 1056), ("q5_0", 32, 300, 2080),
                                       ("q8_0", 5, 4096, 2080), ("q8_0", 31, 8200, 1056),
                                       ("q6k", 4, 257, 256), ("q6kg", 17, 300, 3840), ("q6k", 32, 64, 768)])
def test_wide_gemm_few_rows(ctx, fmt, m, n, k):
    """Up to 32 rows, where the staged forms do not tile K."""
    _check(ctx, fmt, m, n, k, 990 + m)


@pytest.mark.parametrize("m", [3, 4, 20])
def test_wide_set_few_rows_of_mixed_formats(ctx, m):
    """A set of which only the Q6_K matrix (15 super-blocks a row) has no
    staged form: below 4 rows separate products, from there on one wide set."""
    h, n = 3840, 300
    x = np.random.default_rng(8).standard_normal((m, h)).astype(np.float32)
    fmts = ["q4k", "q4k", "q6k"]
    W = [device_weights(ctx, f, n, h, 995 + i) for i, f in enumerate(fmts)]
    ys = [ctx.new_buffer(4 * m * n) for _ in fmts]
    d.gemm_set_f32(ctx, fmts, [w for w, _ in W], ys, [n] * 3, ctx.buffer_from(x), m, h)
    ctx.flush()
    for f, y, (_, raw) in zip(fmts, ys, W):
        ref, sabs = ora.gemv(f, raw, x, n, h)
        check_close(y.read(np.float32, m * n), ref.ravel(), sabs.ravel(), f"{f} of a mixed set of {m} rows")


@pytest.mark.parametrize("m,n,k,wide", [
    (33, 896, 544, False), (128, 896, 1056, False), (64, 2048, 1568, False), (100, 3584, 288, False),
    (8, 3584, 3616, False), (16, 12000, 1568, False), (20, 18944, 544, False), (4, 18944, 2080, False),
    (33, 896, 1088, True), (33, 896, 2080, True), (64, 2560, 544, True), (256, 896, 1056, True),
    (20, 12000, 1056, True), (8, 18944, 2080, True), (8, 8200, 1088, True),
])
def test_q8_0_untiled_k_form(m, n, k, wide):
    """Which Q8_0 GEMMs of a K that the stages do not tile take the wide form in
    a context without switches: not those that the unstaged kernel's few
    workgroups finish sooner."""
    with d.HipContext() as c:
        w, raw = device_weights(c, "q8_0", n, k, 1020 + m)
        x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
        y = c.new_buffer(4 * m * n)
        d.gemm_q8_0_f32(c, w, c.buffer_from(x), y, m, n, k)
        assert d.last_launch_name(c).startswith("k_gemm_q8_0_") != wide, d.last_launch_name(c)
        c.flush()
        rows = [0, m // 2, m - 1]
        ref, sabs = ora.gemv("q8_0", raw, x[rows], n, k)
        check_close(y.read(np.float32, m * n).reshape(m, n)[rows].ravel(), ref.ravel(), sabs.ravel(), f"{m}x{n}x{k}")


@pytest.mark.parametrize("fmt", ["q8_0", "q4kg"])
def test_wide_gemm_whole_and_split_tiles(ctx, fmt):
    """520 tiles: 512 of one workgroup each and 8 with K split (256 compute
    units of two workgroups each), the last one ragged."""
    _check(ctx, fmt, 33, 256 * 519 + 5, 512, 940)


@pytest.mark.parametrize("fmts", [("q4k", "q4k", "q6k"), ("q8_0", "q8_0", "q8_0")])
def test_wide_set_bias(ctx, fmts):
    test_gpu_gemm_set.test_gemm_set_qkv_norm_bias(ctx, fmts, 70)


@pytest.mark.parametrize("fmt,m", [("q4k", 33), ("q8_0", 70)])
def test_wide_set_silu_pair(ctx, fmt, m):
    test_gpu_gemm_set.test_gemm_set_silu_pair(ctx, fmt, m)


@pytest.mark.parametrize("fmt,n,k", [("q6k", 1024, 2048), ("q8_0", 896, 4864), ("q4_0", 1000, 928)])
def test_wide_set_residual(ctx, fmt, n, k):
    test_gpu_gemm_set.test_gemm_set_residual(ctx, fmt, n, k, 70)


def test_wide_set_of_four_and_mixed_pair(ctx):
    """Four matrices of one format (two launches), and a SiLU pair of two
    formats (separate products)."""
    m, h, n = 70, 1024, 300
    x = np.random.default_rng(5).standard_normal((m, h)).astype(np.float32)
    xb = ctx.buffer_from(x)
    W = [device_weights(ctx, "q4k", n, h, 960 + i) for i in range(4)]
    ys = [ctx.new_buffer(4 * m * n) for _ in range(4)]
    d.gemm_set_f32(ctx, ["q4k"] * 4, [w for w, _ in W], ys, [n] * 4, xb, m, h)
    ctx.flush()
    for y, (_, raw) in zip(ys, W):
        ref, sabs = ora.gemv("q4k", raw, x, n, h)
        check_close(y.read(np.float32, m * n), ref.ravel(), sabs.ravel(), "set of four")
    w8, raw8 = device_weights(ctx, "q8_0", n, h, 970)
    d.gemm_set_f32(ctx, ["q4k", "q8_0"], [W[0][0], w8], ys[:2], [n, n], xb, m, h, silu_pair=True)
    ctx.flush()
    g, gs = ora.gemv("q4k", W[0][1], x, n, h)
    u, us = ora.gemv("q8_0", raw8, x, n, h)
    ffn_check(ys[0].read(np.float32, m * n), g.ravel(), gs.ravel(), u.ravel(), us.ravel(), "mixed pair")


def test_wide_qkv_rope_equals_set_then_rope(ctx):
    """As test_gemm_qkv_rope_equals_set_then_rope, at 70 rows: q and keys to
    2e-6 of their range (fused multiply-adds may contract differently), values
    exactly."""
    m, h, hd, heads, kvh, S, start = 70, 1024, 64, 14, 2, 128, 20
    qd, kvd, fmts = heads * hd, kvh * hd, ("q4kg", "q4kg", "q6kg")
    W = [device_weights(ctx, f, n, h, 980 + i)[0] for i, (f, n) in enumerate(zip(fmts, (qd, kvd, kvd)))]
    rng = np.random.default_rng(7)
    x = ctx.buffer_from(rng.standard_normal((m, h)).astype(np.float32))
    gamma = ctx.buffer_from((1 + 0.1 * rng.standard_normal(h)).astype(np.float32))
    biases = [ctx.buffer_from((0.1 * rng.standard_normal(n)).astype(np.float16).view(np.uint16))
              for n in (qd, kvd, kvd)]
    cache0 = rng.standard_normal(kvh * S * hd).astype(np.float32)
    outs = []
    for fused in (True, False):
        q, k, v = (ctx.new_buffer(4 * m * n) for n in (qd, kvd, kvd))
        xn, kc, vc = ctx.new_buffer(4 * m * h), ctx.buffer_from(cache0), ctx.buffer_from(cache0)
        if fused:
            d.gemm_qkv_rope_f32(ctx, fmts, *W, *biases, x, gamma, 1e-6, xn, q, k, v, kc, vc, m, h,
                                qd, kvd, hd, start, 10000.0, S)
        else:
            d.gemm_set_f32(ctx, list(fmts), W, [q, k, v], [qd, kvd, kvd], x, m, h, biases=biases,
                           gamma=gamma, eps=1e-6, xn=xn)
            d.rope_kv_write_batch_f32(ctx, q, k, v, kc, vc, hd, heads, kvh, start, 10000.0, m, S)
        ctx.flush()
        outs.append([b.read(np.float32, n) for b, n in ((q, m * qd), (kc, cache0.size), (vc, cache0.size))])
    for a, b, what in zip(outs[0][:2], outs[1][:2], ("q", "k cache")):
        assert np.max(np.abs(a - b)) <= 2e-6 * np.abs(b).max(), what
    assert np.array_equal(outs[0][2], outs[1][2]), "v cache"


def test_wide_gemm_few_rows_capture():
    """In a context without a workspace, a captured call (and set) of a K that
    nothing tiles runs a GEMV a row as before this form; after an eager call,
    this form; every replay gives the result."""
    m, n, k = 8, 300, 1056
    x = np.random.default_rng(14).standard_normal((m, k)).astype(np.float32)
    with d.HipContext() as ctx:
        W = [device_weights(ctx, "q4_0", n, k, 1010 + i) for i in range(2)]
        xb, ys = ctx.buffer_from(x), [ctx.new_buffer(4 * m * n) for _ in range(2)]
        refs = [ora.gemv("q4_0", raw, x, n, k) for _, raw in W]
        for call, outs in ((lambda: d.gemm_q4_0_f32(ctx, W[0][0], xb, ys[0], m, n, k), 1),
                           (lambda: d.gemm_set_f32(ctx, ["q4_0"] * 2, [w for w, _ in W], ys, [n, n], xb, m, k), 2)):
            for _ in range(2):
                ctx.capture_begin()
                call()
                g = ctx.capture_end()
                for _ in range(2):
                    for y in ys:
                        y.write(np.zeros(m * n, np.float32))
                    g.launch()
                    ctx.flush()
                    for y, (ref, sabs) in list(zip(ys, refs))[:outs]:
                        check_close(y.read(np.float32, m * n), ref.ravel(), sabs.ravel(), "captured")
                    call()
                    ctx.flush()
                del g


def _sized_context(nbytes, former):
    """A context whose workspace holds about nbytes; former: without the wide form."""
    if former:
        os.environ["RUNIT_GEMM_WIDE_WORK"] = str(1 << 62)
    try:
        c = d.HipContext()
    finally:
        os.environ.pop("RUNIT_GEMM_WIDE_WORK", None)
    nrec = nbytes // 4224 | 1  # (the unstaged Q8_0 GEMM takes 4,224 bytes of it a record of 32 rows)
    w, x, y = c.new_buffer(34 * nrec), c.new_buffer(4 * 32 * 32 * nrec), c.new_buffer(4 * 32)
    d.gemm_q8_0_f32(c, w, x, y, 32, 1, 32 * nrec)
    c.flush()
    return c


@pytest.mark.parametrize("what", ["gemm", "set", "pair", "block"])
def test_wide_gemm_capture_in_a_workspace_of_the_staged_form(what):
    """A call that takes the wide form is captured wherever the staged forms
    alone could be, in workspaces from too small for these to enough for both,
    and every replay gives the result."""
    m, h, ff = (70, 1024, 8192) if what == "block" else (70, 2048, 11520)
    rng = np.random.default_rng(15)
    x = rng.standard_normal((m, h if what == "block" else ff)).astype(np.float32)
    accepted = []
    for mb in (2, 4, 5, 6, 7, 8, 10, 12, 16, 24, 40):
        ok = []
        for former in (True, False):
            with _sized_context(mb << 20, former) as c:
                xb = c.buffer_from(x)
                if what == "block":
                    W = [device_weights(c, "q4k", n, k, 1030 + i)[0] for i, (n, k) in enumerate(((h, h), (ff, h), (ff, h), (h, ff)))]
                    at, xm, xn, g, u = (c.new_buffer(4 * m * n) for n in (h, h, h, ff, ff))
                    at.write(0.1 * x)
                    gam = c.buffer_from(np.ones(h, np.float32))
                    out = xb
                    call = lambda: d.gemm_ffn_block_f32(c, ["q4k"] * 4, *W, at, xb, xm, gam, 1e-6, g, u, xn, m, h, h, ff)
                    size = m * h
                else:
                    W = [device_weights(c, "q4k", h, ff, 1040 + i)[0] for i in range(2)]
                    ys = [c.new_buffer(4 * m * h) for _ in range(2)]
                    out, size = ys[0], m * h
                    if what == "gemm":
                        call = lambda: d.gemm_q4k_f32(c, W[0], xb, ys[0], m, h, ff)
                    else:
                        call = lambda: d.gemm_set_f32(c, ["q4k"] * 2, W, ys, [h, h], xb, m, ff, silu_pair=what == "pair")
                c.capture_begin()
                try:
                    call()
                    ok.append(True)
                except d.KernelError:
                    ok.append(False)
                graph = c.capture_end()
                if not ok[-1]:
                    continue
                got = []
                for i in range(3):  # two replays, then eager
                    if what == "block":
                        xb.write(x)
                    else:
                        out.write(np.zeros(size, np.float32))
                    graph.launch() if i < 2 else call()
                    c.flush()
                    got.append(out.read(np.float32, size))
                tol = 1e-5 * np.abs(got[2]).max()  # (the eager call may take the other form)
                assert np.max(np.abs(got[0] - got[2])) <= tol and np.max(np.abs(got[1] - got[2])) <= tol
                del graph
        assert ok[1] or not ok[0], f"{mb} MB: refused"
        accepted.append(ok[1])
    assert accepted[-1] and not accepted[0]


@pytest.fixture(scope="module")
def staged():
    """A context without the wide form for K that the staged forms tile."""
    os.environ["RUNIT_GEMM_WIDE_WORK"] = str(1 << 62)
    try:
        c = d.HipContext()
    finally:
        del os.environ["RUNIT_GEMM_WIDE_WORK"]
    yield c
    c.close()


def _block64(fmts, raws, att, x, gamma, eps, h, qd, ff):
    """The layer after its attention in f64 (projection inputs rounded to f32):
    x_mid and x with the Σ|w·x| of the O and down sums."""
    y, so = ora.gemv(fmts[0], raws[0], att, h, qd)
    xm = x + y
    xn = xm / np.sqrt((xm * xm).mean(1, keepdims=True) + eps) * gamma
    g, _ = ora.gemv(fmts[1], raws[1], xn, ff, h)
    u, _ = ora.gemv(fmts[2], raws[2], xn, ff, h)
    y, sd = ora.gemv(fmts[3], raws[3], g / (1 + np.exp(-g)) * u, h, ff)
    return xm, so, xm + y, sd


def _check_block(ctx, staged, fmts, m, h, qd, ff, call, att, rows, seed):
    """call(context, weights, x, x_mid, gamma, eps, g, u, xn) on both contexts:
    x_mid within 1e-6 of its sums (as the GEMMs above) and its own rounding, x
    within 1e-5 of the down sums (the product silu(gate)·up carries the error of
    its own two sums, some ten times smaller than they), and other bits than the
    staged forms': the wide ones ran."""
    x0 = np.random.default_rng(seed).standard_normal((m, h)).astype(np.float32)
    gamma = np.linspace(0.5, 1.5, h, dtype=np.float32)
    outs = []
    for c in (ctx, staged):
        W = [device_weights(c, f, n, k, seed + i)
             for i, (f, n, k) in enumerate(zip(fmts, (h, ff, ff, h), (qd, h, h, ff)))]
        x, xm = c.buffer_from(x0), c.new_buffer(4 * m * h)
        g, u, xn = c.new_buffer(4 * m * ff), c.new_buffer(4 * m * ff), c.new_buffer(4 * m * h)
        call(c, [w for w, _ in W], x, xm, c.buffer_from(gamma), 1e-6, g, u, xn)
        c.flush()
        outs.append((xm.read(np.float32, m * h).reshape(m, h), x.read(np.float32, m * h).reshape(m, h)))
    xm, so, x, sd = _block64(fmts, [r for _, r in W], att[rows], x0[rows], gamma, 1e-6, h, qd, ff)
    for got, ref, s, tol, what in ((outs[0][0], xm, so, 1e-6, "x_mid"), (outs[0][1], x, sd, 1e-5, "x")):
        err = np.abs(got[rows] - ref)
        bound = tol * s + 2.0 ** -23 * np.abs(ref)
        assert np.all(err <= bound), f"{what}: {(err / bound).max():.2f} of the bound"
        assert np.all(np.isfinite(got)), what
    if h % 128 == 0:  # (the staged forms tile it)
        assert not np.array_equal(outs[0][0], outs[1][0]) and not np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("fmts,m,h,qd,ff", [
    (("q4k", "q4k", "q4k", "q6k"), 33, 1024, 1024, 2048),
    (("q8_0", "q8_0", "q8_0", "q8_0"), 65, 1056, 1120, 2592),  # (K that nothing else tiles, on both)
    (("q8_0", "q8_0", "q8_0", "q8_0"), 65, 896, 4608, 2560),   # preparations of up to and over 4,096
    (("q4kg", "q4kg", "q4kg", "q6kg"), 130, 4352, 512, 5120),
    (("q4k", "q4k", "q4k", "q4k"), 440, 20480, 512, 512),      # O: 560 tiles, 512 of them whole
])
def test_wide_block(ctx, staged, fmts, m, h, qd, ff):
    att = np.random.default_rng(m).standard_normal((m, qd)).astype(np.float32)

    def call(c, W, x, xm, gamma, eps, g, u, xn):
        d.gemm_ffn_block_f32(c, fmts, *W, c.buffer_from(att), x, xm, gamma, eps, g, u, xn, m, h, qd, ff)

    _check_block(ctx, staged, fmts, m, h, qd, ff, call, att, [0, m // 2, m - 1], 1050 + m)


@pytest.mark.parametrize("fmts,hd,heads,kvh,m,start", [
    (("q4k", "q4k", "q4k", "q6k"), 128, 8, 2, 33, 300),
    (("q8_0", "q8_0", "q8_0", "q8_0"), 64, 14, 2, 70, 200),
    (("q4kg", "q4kg", "q4kg", "q6kg"), 128, 36, 4, 34, 200),   # O's K of 4,608
])
def test_wide_block_with_folded_attention(ctx, staged, fmts, hd, heads, kvh, m, start):
    """The attention's key-range partials merged in the wide form's preparation."""
    h, qd, ff, S = 768, heads * hd, 1536, start + m
    rng = np.random.default_rng(m)
    q = rng.standard_normal((m, qd)).astype(np.float32)
    kc, vc = (rng.standard_normal((kvh, S, hd)).astype(np.float32) for _ in range(2))
    att = ora.causal_attention(q, kc, vc, m, heads, kvh, hd, S, S, start).reshape(m, qd)

    def call(c, W, x, xm, gamma, eps, g, u, xn):
        at = c.buffer_from(np.full(m * qd, 7.0, np.float32))
        d.gemm_attn_ffn_block_f32(c, c.buffer_from(q), c.buffer_from(kc), c.buffer_from(vc), S, heads, kvh, hd, S,
                                  start, at, fmts, *W, x, xm, gamma, eps, g, u, xn, m, h, ff)
        c.flush()
        assert np.all(at.read(np.float32, m * qd) == 7.0)  # (the folded form does not write it)

    _check_block(ctx, staged, fmts, m, h, qd, ff, call, att, [0, m // 2, m - 1], 1060 + m)


@pytest.mark.parametrize("what", ["bias", "rope", "pair", "residual"])
def test_wide_set_whole_and_split_tiles(ctx, staged, what):
    """Sets of 520 tiles and more, 512 of one workgroup each, the others with K
    split: the sums of the split ones alone are added, in 16-byte units (rows of
    a multiple of 4), against the oracle and with other bits than the staged
    form's."""
    m, k, hd = 35, 512, 64
    ns = {"bias": [256 * 400, 256 * 100 + 4, 256 * 19 + 8], "rope": [256 * 400, 256 * 100 + 64, 256 * 19 + 64],
          "pair": [128 * 519 + 4] * 2, "residual": [256 * 519 + 4]}[what]
    if what == "rope":
        ns[2] = ns[1]
    rng = np.random.default_rng(16)
    x = rng.standard_normal((m, k)).astype(np.float32)
    biases = [(0.1 * rng.standard_normal(n)).astype(np.float16) for n in ns]
    rows, outs = [0, m - 1], []
    for c in (ctx, staged):
        W = [device_weights(c, "q8_0", n, k, 1070 + i) for i, n in enumerate(ns)]
        xb, ys = c.buffer_from(x), [c.new_buffer(4 * m * n) for n in ns]
        bb = [c.buffer_from(b.view(np.uint16)) for b in biases]
        if what == "rope":
            kvh = ns[1] // hd
            xn, kc, vc = c.new_buffer(4 * m * k), *(c.new_buffer(4 * kvh * m * hd) for _ in range(2))
            gam = c.buffer_from(np.ones(k, np.float32))
            d.gemm_qkv_rope_f32(c, ["q8_0"] * 3, *[w for w, _ in W], *bb, xb, gam, 0.0, xn, *ys, kc, vc, m, k, *ns[:2],
                                hd, 0, 10000.0, m)
            c.flush()
            x = xn.read(np.float32, m * k).reshape(m, k)
            got = [ys[0].read(np.float32, m * ns[0]).reshape(m, -1)] + [
                b.read(np.float32, kvh * m * hd).reshape(kvh, m, hd).transpose(1, 0, 2).reshape(m, -1) for b in (kc, vc)]
        else:
            kw = {"bias": dict(biases=bb), "pair": dict(silu_pair=True),
                  "residual": dict(res=c.buffer_from(np.tile(biases[0].astype(np.float32), (m, 1))))}[what]
            d.gemm_set_f32(c, ["q8_0"] * len(ns), [w for w, _ in W], ys, ns, xb, m, k, **kw)
            c.flush()
            got = [y.read(np.float32, m * n).reshape(m, n) for y, n in zip(ys, ns)][:1 if what == "pair" else 3]
        outs.append(got)
    refs = [ora.gemv("q8_0", raw, x[rows], n, k) for (_, raw), n in zip(W, ns)]
    if what == "pair":
        ffn_check(outs[0][0][rows].ravel(), refs[0][0].ravel(), refs[0][1].ravel(), refs[1][0].ravel(),
                  refs[1][1].ravel(), what)
    else:
        for i, (g, (ref, sabs), b) in enumerate(zip(outs[0], refs, biases)):
            ref = ref + b.astype(np.float64)
            if what == "rope" and i < 2:  # pairs (j, j + 32) of each head, row r at position r
                a = np.array(rows)[:, None, None] / 10000.0 ** (2 * np.arange(32) / hd)
                t = ref.reshape(2, -1, 2, 32)
                ref = np.stack([t[:, :, 0] * np.cos(a) - t[:, :, 1] * np.sin(a),
                                t[:, :, 0] * np.sin(a) + t[:, :, 1] * np.cos(a)], 2).reshape(2, -1)
                sabs = np.repeat(sabs.reshape(2, -1, 2, 32).sum(2, keepdims=True), 2, 2).reshape(2, -1)
                sabs += np.abs(ref).max()  # (angles of up to 34 radians in f32: 4e-6 of the pair)
            check_close(g[rows].ravel(), ref.ravel(), sabs.ravel(), f"{what} {i}", extra=1e-6 * np.abs(ref).ravel())
    assert any(not np.array_equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("fmt,m,n,k,wide", [
    ("q8_0", 124, 3584, 3584, False), ("q8_0", 125, 3584, 3584, True),
    ("q4k", 32, 18944, 3584, False), ("q4k", 33, 18944, 3584, True),
    ("q8_0", 192, 8192, 1024, False), ("q8_0", 256, 8192, 1024, True),       # short K of 32-element blocks
    ("q4_0", 160, 12000, 1024, False), ("q4_0", 192, 12000, 1024, True),
    ("q4_0g", 128, 13928, 2048, False), ("q4_0g", 256, 13928, 2048, True), ("q5_0", 65, 10000, 2560, True),
    ("q4k", 96, 18944, 2048, False), ("q4k", 97, 18944, 2048, True), ("q8_0", 65, 18944, 1536, False),
])
def test_wide_gemm_rule(ctx, staged, fmt, m, n, k, wide):
    """Which GEMMs of a K that the staged forms tile take the wide form in a
    context without switches: from 33 rows and 1.6e9 rows x weights on, more
    where the staged form stays ahead longer.  The result is that form's, bit
    for bit."""
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float32)
    outs = []
    with d.HipContext() as plain:
        for c in (plain, ctx, staged):
            w, _ = device_weights(c, fmt, n, k, 1080)
            y = c.new_buffer(4 * m * n)
            getattr(d, f"gemm_{fmt}_f32")(c, w, c.buffer_from(x), y, m, n, k)
            c.flush()
            outs.append(y.read(np.float32, m * n))
    assert np.array_equal(outs[0], outs[1 if wide else 2])
    assert m <= 32 or not np.array_equal(outs[1], outs[2])


@pytest.mark.parametrize("fmt,m,h,ff,wide", [("q8_0", 96, 1536, 4096, False), ("q8_0", 192, 1536, 4096, True),
                                             ("q4_0g", 224, 1024, 4096, False), ("q4_0g", 320, 1024, 4096, True),
                                             ("q4k", 33, 2048, 8192, True)])
def test_wide_block_rule(ctx, staged, fmt, m, h, ff, wide):
    """The same of layer blocks."""
    rng = np.random.default_rng(m)
    x, att = (rng.standard_normal((m, h)).astype(np.float32) for _ in range(2))
    outs = []
    with d.HipContext() as plain:
        for c in (plain, ctx, staged):
            W = [device_weights(c, fmt, n, k, 1090 + i)[0] for i, (n, k) in enumerate(((h, h), (ff, h), (ff, h), (h, ff)))]
            xb, xm, xn, g, u = c.buffer_from(x), *(c.new_buffer(4 * m * n) for n in (h, h, ff, ff))
            d.gemm_ffn_block_f32(c, [fmt] * 4, *W, c.buffer_from(att), xb, xm, c.buffer_from(np.ones(h, np.float32)),
                                 1e-6, g, u, xn, m, h, h, ff)
            c.flush()
            outs.append(xb.read(np.float32, m * h))
    assert np.array_equal(outs[0], outs[1 if wide else 2])
    assert not np.array_equal(outs[1], outs[2])


@pytest.mark.parametrize("fmts,m,h,ff,sets", [(("q4k", "q4k", "q4k", "q6k"), 4, 768, 2304, True),
                                              (("q4k", "q4k", "q4k", "q6k"), 5, 768, 2304, False),
                                              (("q8_0",) * 4, 64, 96, 288, True), (("q8_0",) * 4, 64, 160, 480, False)])
def test_wide_block_of_untiled_k_or_its_sets(fmts, m, h, ff, sets):
    """4 rows, and hidden sizes below 160, run as the three sets, in their launches."""
    x = np.random.default_rng(m).standard_normal((m, h)).astype(np.float32)
    counts, outs = [], []
    with d.HipContext() as c:
        W = [device_weights(c, f, n, k, 1100 + i)[0] for i, (f, n, k) in enumerate(zip(fmts, (h, ff, ff, h), (h, h, h, ff)))]
        gam = c.buffer_from(np.ones(h, np.float32))
        for block in (True, False):
            at, xb, xm, xn, g, u = (c.buffer_from(np.ones((m, n), np.float32)) for n in (h, h, h, h, ff, ff))
            xb.write(x)
            n0 = d.launch_count(c)
            if block:
                d.gemm_ffn_block_f32(c, fmts, *W, at, xb, xm, gam, 1e-6, g, u, xn, m, h, h, ff)
            else:
                d.gemm_set_f32(c, fmts[:1], W[:1], [xm], [h], at, m, h, res=xb)
                d.gemm_set_f32(c, fmts[1:3], W[1:3], [g, u], [ff, ff], xm, m, h, gamma=gam, eps=1e-6, xn=xn, silu_pair=True)
                d.gemm_set_f32(c, fmts[3:], W[3:], [xb], [h], g, m, ff, res=xm)
            counts.append(d.launch_count(c) - n0)
            c.flush()
            outs.append(xb.read(np.float32, m * h))
    assert (counts[0] == counts[1]) == sets, counts
    assert np.max(np.abs(outs[0] - outs[1])) <= 1e-5 * np.abs(outs[1]).max()
