"""The long-prompt attention (k_attn_pf_f32_hd64 / 128) against the oracle's
causal attention: the edges of its 128-column workgroups and 32-position
records, positions split over workgroups, sequences of a batch, keys and
values of magnitudes far apart, infinities.  Tolerance: a convex combination
of values with an f32 softmax, 1e-5 of the value range (test_gpu_verify)."""
import os

import numpy as np
import pytest

import oracle_lib as ora
from runit_mac_amd import dispatch as d

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    """A context whose attention takes this form however short the prompt."""
    os.environ["RUNIT_ATTN_PF_WORK"] = "0"
    try:
        c = d.HipContext()
    finally:
        del os.environ["RUNIT_ATTN_PF_WORK"]
    yield c
    c.close()


def run(ctx, q, kc, vc, batch, M, kv_len, H, KVH, hd, S, q_start):
    bo = ctx.new_buffer(4 * (batch * M * H * hd + 64))
    bo.write(np.full(batch * M * H * hd + 64, 7.0, np.float32))
    d.flash_attention_f32(ctx, ctx.buffer_from(q), ctx.buffer_from(kc), ctx.buffer_from(vc), bo, batch, M, kv_len, H,
                          KVH, hd, S, q_start)
    assert d.last_launch_name(ctx) in (f"k_attn_pf_f32_hd{hd}", f"k_attn_pf_merge_hd{hd}")
    ctx.flush()
    got = bo.read(np.float32, batch * M * H * hd + 64)
    assert np.all(got[batch * M * H * hd:] == 7.0), "past the last row"
    return got[:batch * M * H * hd].reshape(batch, M, H * hd)


@pytest.mark.parametrize("hd,H,KVH,M,kv_len,q_start", [
    (64, 1, 1, 1, 1, 0),          # one query, one position
    (128, 2, 2, 33, 33, 0),       # one column block, the second record of one position
    (64, 14, 2, 19, 200, 181),    # 133 columns: a second block of 5
    (128, 28, 4, 40, 300, 260),   # position ranges merged
    (64, 8, 8, 130, 130, 0),      # ranges that the first block does not see
    (128, 6, 2, 50, 64, 30),      # rows past kv_len: all of it
    (64, 4, 2, 300, 1000, 700),
])
def test_prefill_attention(ctx, hd, H, KVH, M, kv_len, q_start):
    rng = np.random.default_rng(hd + M + kv_len)
    S = kv_len + 16
    q = rng.standard_normal(M * H * hd).astype(np.float32)
    kc, vc = (rng.standard_normal(KVH * S * hd).astype(np.float32) for _ in range(2))
    # past the last position that a query sees the cache is not read
    last = min(kv_len, q_start + M)
    for x in (kc, vc):
        x.reshape(KVH, S, hd)[:, last:] = np.nan
    got = run(ctx, q, kc, vc, 1, M, kv_len, H, KVH, hd, S, q_start)[0]
    ref = ora.causal_attention(q, kc, vc, M, H, KVH, hd, kv_len, S, q_start)
    assert np.max(np.abs(got - ref)) <= 1e-5 * np.nanmax(np.abs(vc))


def test_prefill_attention_batch(ctx):
    rng = np.random.default_rng(9)
    hd, H, KVH, M, kv_len, S = 64, 6, 2, 50, 300, 310
    q = rng.standard_normal(2 * M * H * hd).astype(np.float32)
    kc, vc = (rng.standard_normal(2 * KVH * S * hd).astype(np.float32) for _ in range(2))
    got = run(ctx, q, kc, vc, 2, M, kv_len, H, KVH, hd, S, kv_len - M)
    per = KVH * S * hd
    for b in range(2):
        ref = ora.causal_attention(q.reshape(2, -1)[b], kc[b * per:(b + 1) * per], vc[b * per:(b + 1) * per], M, H,
                                   KVH, hd, kv_len, S, kv_len - M)
        assert np.max(np.abs(got[b] - ref)) <= 1e-5 * np.abs(vc).max(), b


def test_prefill_attention_scales(ctx):
    """Keys, queries and values whose magnitudes differ by 2^40 from row to
    row (scores of every size, exponents of records rising and falling), and
    all-zero rows: the error of each output within 1e-5 of the values its
    query weights, Σ p·|v|."""
    rng = np.random.default_rng(11)
    hd, H, KVH, M, S = 128, 2, 1, 70, 200
    q = rng.standard_normal((M, H, hd)).astype(np.float32)
    kc = rng.standard_normal((S, hd)).astype(np.float32)
    vc = rng.standard_normal((S, hd)).astype(np.float32)
    q *= np.exp2(rng.integers(-20, 1, (M, 1, 1))).astype(np.float32)
    kc *= np.exp2(rng.integers(-20, 1, (S, 1))).astype(np.float32)
    vc *= np.exp2(rng.integers(-20, 21, S // 8).repeat(8)[:, None]).astype(np.float32)
    vc[40:80] *= 2.0 ** -60
    q[3], kc[5], vc[64:96] = 0, 0, 0
    got = run(ctx, q.ravel(), kc.ravel(), vc.ravel(), 1, M, S, H, KVH, hd, S, S - M)[0]
    ref = ora.causal_attention(q.ravel(), kc.ravel(), vc.ravel(), M, H, KVH, hd, S, S, S - M)
    mag = ora.causal_attention(q.ravel(), kc.ravel(), np.abs(vc).ravel(), M, H, KVH, hd, S, S, S - M)
    assert np.all(np.abs(got - ref) <= 1e-5 * mag)


def check_values(ctx, q, kc, vc, M, H, KVH, hd, S, q_start):
    """Each output within 1e-5 of the values that its query weights, Σ p·|v|."""
    args = (M, H, KVH, hd, S, S, q_start)
    got = run(ctx, q.ravel(), kc.ravel(), vc.ravel(), 1, M, S, H, KVH, hd, S, q_start)[0]
    ref = ora.causal_attention(q.ravel(), kc.ravel(), vc.ravel(), *args)
    mag = ora.causal_attention(q.ravel(), kc.ravel(), np.abs(vc).ravel(), *args)
    err = np.abs(got - ref)
    assert np.all(err <= 1e-5 * mag), f"{(err / np.maximum(mag, 1e-300)).max():.1e}"


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("r", [10, 16, 24, 32, 60, -30])
def test_prefill_attention_outweighed_values(ctx, hd, r):
    """Values 2^r times the others' whose softmax weight is e^-20·2^-r: in a
    record of their own at the start, and beside others at the end of one."""
    rng = np.random.default_rng(20 + abs(r))
    H, KVH, M, S = 2, 1, 40, 500
    q, kc, vc = (rng.standard_normal((n, hd)).astype(np.float32) for n in (M * H, S, S))
    q[:, 0], kc[:, 0] = np.sqrt(hd), 0
    for at in (slice(0, 32), slice(440, 448)):
        kc[at, 0] = -20 - max(r, 0) * np.log(2)
        vc[at] *= np.float32(2.0 ** r)
    check_values(ctx, q, kc, vc, M, H, KVH, hd, S, S - M)


@pytest.mark.parametrize("std", [1.0, 1e-2, 1e-6, 1e-30])
def test_prefill_attention_zero_values(ctx, std):
    """Records and single positions of all-zero values (padding) among small ones."""
    rng = np.random.default_rng(21)
    hd, H, KVH, M, S = 64, 4, 2, 50, 410
    q, kc, vc = (rng.standard_normal((n, hd)).astype(np.float32) for n in (M * H, KVH * S, KVH * S))
    vc = (vc * std).astype(np.float32).reshape(KVH, S, hd)
    vc[:, :32] = vc[:, 96:160] = vc[:, 330] = 0
    check_values(ctx, q, kc, vc, M, H, KVH, hd, S, S - M)


@pytest.mark.parametrize("r", [24, 40, 100])
def test_prefill_attention_large_later_values(ctx, r):
    """A value of 2^r leaves the queries before it, in its record too, as they are."""
    rng = np.random.default_rng(22)
    hd, H, KVH, M = 128, 2, 1, 70
    q, kc, vc = (rng.standard_normal((n, hd)).astype(np.float32) for n in (M * H, M, M))
    vc[31] *= np.float32(2.0 ** r)
    check_values(ctx, q, kc, vc, M, H, KVH, hd, M, 0)


def test_prefill_attention_infinities(ctx):
    """A key of -inf score leaves its position out, one of +inf makes the rows
    that see it NaN, an infinite value its element infinite: as in f32
    throughout; rows that do not see them are untouched."""
    rng = np.random.default_rng(12)
    hd, H, KVH, M, S = 64, 2, 1, 90, 100
    q = np.abs(rng.standard_normal((M, H, hd))).astype(np.float32)
    kc, vc = (rng.standard_normal((S, hd)).astype(np.float32) for _ in range(2))
    clean = (q.ravel(), kc.copy(), vc.copy())
    kc[20, 7] = -np.inf
    kc[70, 3] = np.inf
    vc[45, 9] = np.inf
    got = run(ctx, q.ravel(), kc.ravel(), vc.ravel(), 1, M, M, H, KVH, hd, S, 0)[0].reshape(M, H, hd)
    low = clean[1].copy()
    low[20] = -1e4 * np.ones(hd)  # (a score below every other by far)
    for lo, hi, keys in ((0, 20, clean[1]), (20, 70, low)):
        ref = ora.causal_attention(clean[0], keys.ravel(), clean[2].ravel(), M, H, KVH, hd, M, S, 0).reshape(M, H, hd)
        for r in range(lo, hi):
            e = np.arange(hd) != 9 if r >= 45 else np.ones(hd, bool)  # (the rows before 45 share its record)
            assert np.max(np.abs(got[r][:, e] - ref[r][:, e])) <= 1e-5 * np.abs(clean[2]).max(), r
    assert np.all(np.isinf(got[45:70, :, 9]))
    assert np.all(np.isnan(got[70:]))


@pytest.mark.parametrize("what", ["range", "outweighed key", "outweighed value"])
def test_prefill_attention_nan_ranges(ctx, what):
    """A NaN reaches every query that sees it, whatever the weight of the range
    of positions that holds it (520 positions: ranges of 128): a range of NaN
    keys, a NaN key and an infinite value (0·inf) beside keys of scores below
    all others by 300."""
    rng = np.random.default_rng(23)
    hd, H, KVH, M, S = 64, 2, 1, 40, 520
    q, kc, vc = (rng.standard_normal((n, hd)).astype(np.float32) for n in (M * H, S, S))
    q[:, 0], kc[:, 0] = np.sqrt(hd), 0
    kc[128:256, 0] = -300
    ref = ora.causal_attention(q.ravel(), kc.ravel(), vc.ravel(), M, H, KVH, hd, S, S, S - M).reshape(M * H, hd)
    element = np.ones(hd, bool)
    if what == "range":
        kc[128:256] = np.nan
    elif what == "outweighed key":
        kc[130] = np.nan
    else:
        vc[130, 9] = np.inf
        element = np.arange(hd) == 9
    got = run(ctx, q.ravel(), kc.ravel(), vc.ravel(), 1, M, S, H, KVH, hd, S, S - M)[0].reshape(M * H, hd)
    assert np.all(np.isnan(got[:, element]))
    assert np.all(np.abs(got - ref)[:, ~element] <= 1e-5 * np.abs(vc[:, ~element]).max(initial=0))


def test_prefill_attention_capture():
    """Captured in a context whose workspace is not sized the call keeps the
    kernel that needs none; after an eager call it is captured in this form,
    and replays after eager work of its own give the eager result."""
    hd, H, KVH, M, S = 64, 14, 2, 300, 300
    rng = np.random.default_rng(13)
    q = rng.standard_normal(M * H * hd).astype(np.float32)
    kc, vc = (rng.standard_normal(KVH * S * hd).astype(np.float32) for _ in range(2))
    os.environ["RUNIT_ATTN_PF_WORK"] = "0"
    try:
        ctx = d.HipContext()
    finally:
        del os.environ["RUNIT_ATTN_PF_WORK"]
    with ctx:
        bufs = [ctx.buffer_from(a) for a in (q, kc, vc)]
        bo = ctx.new_buffer(4 * M * H * hd)
        call = lambda: d.flash_attention_f32(ctx, *bufs, bo, 1, M, S, H, KVH, hd, S, 0)
        ref = ora.causal_attention(q, kc, vc, M, H, KVH, hd, S, S, 0)
        for kernel in (f"k_attn_mq_f32_hd{hd}", f"k_attn_pf_merge_hd{hd}"):
            ctx.capture_begin()
            call()
            g = ctx.capture_end()
            assert d.last_launch_name(ctx) == kernel
            for _ in range(3):
                bo.write(np.zeros(M * H * hd, np.float32))
                g.launch()
                ctx.flush()
                got = bo.read(np.float32, M * H * hd).reshape(M, H * hd)
                assert np.max(np.abs(got - ref)) <= 1e-5 * np.abs(vc).max()
                call()  # (eager; sizes the workspace the first time)
                ctx.flush()
            del g


@pytest.mark.parametrize("hd,H,KVH,batch,M,start,form", [
    (128, 28, 4, 1, 512, 1536, "pf"),
    (64, 14, 2, 1, 300, 1000, "pf"),
    (128, 28, 4, 4, 32, 2000, "pf"),
    (128, 28, 4, 1, 300, 500, "mq"),    # fewer than 1,024 positions
    (64, 14, 2, 1, 64, 4000, "mq"),     # few columns of a KV head
    (128, 28, 4, 1, 16, 8192, "mq"),
    (64, 8, 8, 16, 8, 4000, "mq"),
    (128, 28, 4, 8, 4, 4092, "mq"),
])
def test_prefill_attention_rule(hd, H, KVH, batch, M, start, form):
    """Which calls of a context without switches take this form: not those of
    few queries a sequence, whose caches its preparation would rewrite for
    little (k_attn_mq is up to four times as fast there)."""
    S = start + M
    with d.HipContext() as ctx:
        bufs = [ctx.buffer_from(np.ones(n, np.float32)) for n in (batch * M * H * hd, batch * KVH * S * hd)]
        bo = ctx.new_buffer(4 * batch * M * H * hd)
        d.flash_attention_f32(ctx, bufs[0], bufs[1], bufs[1], bo, batch, M, S, H, KVH, hd, S, start)
        ctx.flush()
        assert d.last_launch_name(ctx).startswith(f"k_attn_{form}_")
        assert np.max(np.abs(bo.read(np.float32, batch * M * H * hd) - 1)) <= 1e-5


def test_prefill_attention_rules_own_range():
    """A prompt chunk that takes this form without switches, against the oracle."""
    rng = np.random.default_rng(24)
    hd, H, KVH, M, S, start = 64, 14, 2, 300, 1300, 1000
    q = rng.standard_normal(M * H * hd).astype(np.float32)
    kc, vc = (rng.standard_normal(KVH * S * hd).astype(np.float32) for _ in range(2))
    with d.HipContext() as c:
        got = run(c, q, kc, vc, 1, M, S, H, KVH, hd, S, start)[0]
    ref = ora.causal_attention(q, kc, vc, M, H, KVH, hd, S, S, start)
    assert np.max(np.abs(got - ref)) <= 1e-5 * np.abs(vc).max()
