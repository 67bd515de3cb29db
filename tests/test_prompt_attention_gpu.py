"""Prompts over both caches in the form for many columns (128 (token, head) columns a workgroup, 32 a wave): partly filled workgroups and waves, blocks that
only some waves see, every way the results leave by, and scores at the ends of the range."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D = 128
SCALE = 1.0 / np.sqrt(D)


@pytest.fixture(scope="module")
def xh():
    from xfastertransformer_amd import capi
    capi.init(0)
    return capi


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _cache(xh, orc, k, v, int8=0):
    """k, v: [B, tokens, H * D]"""
    B, n, w = k.shape
    kc, vc = orc.KVCache(int8, B, w // D, n, D), orc.KVCache(int8, B, w // D, n, D)
    for b in range(B):
        kc.store(b, 0, k[b])
        vc.store(b, 0, v[b])
    dc = xh.KVCache(xh.INT8 if int8 else xh.FP16, B, w // D, n, D)
    dc.load(0, kc.data, kc.scales)
    dc.load(1, vc.data, vc.scales)
    return kc, vc, dc


def _attend(xh, orc, dc, q, B, S, qh, past, out_dtype, pitch, skip, scale=SCALE):
    """Results at `skip` elements from a 256-byte border, rows `pitch` elements apart; what lies between the rows stays as it is."""
    rows, width, bf16 = q.shape[0], q.shape[1], out_dtype == xh.BF16
    qd = xh.DeviceBuffer.from_numpy(orc.to_bf16(q))
    mark = np.full(rows * pitch + skip, 7.0, np.float32)
    od = xh.DeviceBuffer.from_numpy(orc.to_bf16(mark) if bf16 else mark)
    at = C.c_void_p(od.ptr.value + skip * (2 if bf16 else 4))
    xh.attention(dc, qd.ptr, width, at, pitch, out_dtype, B, S, qh, scale, past)
    xh.synchronize()
    out = od.to_numpy(np.uint16, mark.shape) if bf16 else od.to_numpy(np.float32, mark.shape)
    out = (orc.from_bf16(out) if bf16 else out)
    assert (out[:skip] == 7.0).all()
    out = out[skip:].reshape(rows, pitch)
    assert (out[:, width:] == 7.0).all()
    return out[:, :width]


@pytest.mark.parametrize("B,S,past,qh,kvh,kind,extra,skip", [
    (1, 512, 0, 32, 8, "bf16", 0, 0),  # whole workgroups
    (1, 521, 0, 32, 8, "bf16", 8, 8),  # a last workgroup of 36 columns: one wave full, one of 4, two without any
    (1, 517, 31, 32, 8, "bf16", 4, 4),  # rows on 8-byte borders
    (1, 517, 32, 32, 8, "bf16", 1, 1),  # rows on 2-byte borders
    (2, 300, 1, 32, 8, "f32", 4, 0),
    (16, 33, 0, 32, 32, "bf16", 0, 0),  # one head a group: a wave's columns are 32 tokens
    (9, 257, 95, 8, 8, "f32", 0, 4),
    (64, 2, 700, 128, 4, "bf16", 0, 0),  # a token's heads fill a wave; the first three blocks lie before all new tokens
    (5, 129, 64, 28, 4, "bf16", 8, 0),  # 7 heads a group: waves begin inside a token
])
def test_columns_and_ways_out(xh, orc, B, S, past, qh, kvh, kind, extra, skip):
    rng = np.random.default_rng(S * 31 + past)
    k, v = (rng.standard_normal((B, past + S, kvh * D)).astype(np.float32) for _ in range(2))
    kc, vc, dc = _cache(xh, orc, k, v)
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)))
    got = _attend(xh, orc, dc, q, B, S, qh, past, xh.BF16 if kind == "bf16" else xh.F32, qh * D + extra, skip)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, [past] * B, SCALE)
    # fp16 probabilities: 2^-11 of a value each; bf16 results 2^-9 on top
    assert (np.abs(got - ref) <= 3e-3 + np.abs(ref) * (2.0 ** -8 if kind == "bf16" else 0.0)).all(), np.abs(got - ref).max()
    dc.free()


@pytest.mark.parametrize("B,S,past,qh,kvh", [
    (7, 70, 0, 36, 9),  # 63 (sequence, KV head) pairs, 8 a group: bands of 3 and 5 groups, the last group of 7 pairs
    (11, 130, 40, 16, 8),  # 11 groups: bands of 1, 5 and 5
    (10, 65, 3, 32, 8),  # 10: whole bands only
    (3, 300, 0, 24, 3),  # 9 pairs in two groups
    (13, 66, 0, 20, 5),  # 65 pairs: 9 groups, the last of one pair
])
@pytest.mark.parametrize("int8", [0, 1])
def test_bands_of_pairs(xh, orc, B, S, past, qh, kvh, int8):
    """Every pair's every column group is walked whatever the number of pairs; tolerance as above, an INT8 cache's values as it holds them."""
    rng = np.random.default_rng(B * S)
    k, v = (rng.standard_normal((B, past + S, kvh * D)).astype(np.float32) for _ in range(2))
    kc, vc, dc = _cache(xh, orc, k, v, int8)
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)))
    got = _attend(xh, orc, dc, q, B, S, qh, past, xh.BF16, qh * D, 0)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, [past] * B, SCALE)
    assert (np.abs(got - ref) <= 3e-3 + np.abs(ref) * 2.0 ** -8).all(), np.abs(got - ref).max()
    dc.free()


@pytest.mark.parametrize("score", [-1e30, -3000.0, 3000.0, 1e30])
def test_scores_at_the_ends_of_the_range(xh, orc, score):
    """The first 40 tokens score minus infinity, far below all others (the first blocks' weights vanish once others are seen), far above them (the others' do)
    or NaN-making plus infinity with every query; a NaN among the last token's values stays with the queries that see it."""
    S, qh, kvh = 600, 32, 8
    rng = np.random.default_rng(3)
    k, v = (rng.standard_normal((1, S, kvh * D)).astype(np.float32) for _ in range(2))
    k.reshape(S, kvh, D)[:40, :, 0] = score
    k.reshape(S, kvh, D)[40:, :, 0] = 0.0
    v[0, S - 1, 5] = np.nan
    kc, vc, dc = _cache(xh, orc, k, v)
    q = orc.round_bf16(rng.standard_normal((S, qh * D)))
    q.reshape(S, qh, D)[:, :, 0] = 1.0
    got = _attend(xh, orc, dc, q, 1, S, qh, 0, xh.F32, qh * D, 0).reshape(S, qh, D)
    kf, vf = (c.as_f32()[0].transpose(1, 0, 2).astype(np.float64) for c in (kc, vc))  # [tokens, heads, D]
    if score == 1e30:  # plus infinity minus plus infinity
        assert np.isnan(got).all()
        return
    for i in (0, 39, 40, 41, 100, 311, 575):
        with np.errstate(invalid="ignore"):
            x = np.einsum("hd,thd->ht", q.reshape(S, qh, D)[i].astype(np.float64), np.repeat(kf[:i + 1], qh // kvh, 1)) * SCALE
            w = np.exp(x - x.max(1, keepdims=True))
            ref = np.einsum("ht,thd->hd", w / w.sum(1, keepdims=True), np.repeat(vf[:i + 1], qh // kvh, 1))
        if score == -1e30 and i < 40:
            assert np.isnan(got[i]).all()  # nothing but minus infinity
        else:
            assert np.abs(got[i] - ref).max() < 3e-3, (i, np.abs(got[i] - ref).max())
    # (a token of the same 32-token block takes part with a weight of zero: only the queries of earlier blocks are sure to be free of it)
    assert np.isfinite(got[41:576]).all() and np.isnan(got[S - 1]).any()
    dc.free()


@pytest.mark.parametrize("B,S,past,qh,kvh,kind,extra,skip", [
    (1, 512, 0, 32, 8, "bf16", 0, 0),
    (1, 521, 0, 32, 8, "bf16", 8, 8),
    (1, 517, 31, 32, 8, "bf16", 1, 1),
    (2, 300, 1, 32, 8, "f32", 4, 0),
    (16, 33, 0, 32, 32, "bf16", 0, 0),  # two blocks, the second with one token
    (33, 31, 0, 32, 32, "f32", 0, 0),  # a single block
    (12, 65, 0, 32, 32, "bf16", 4, 4),  # three
    (64, 2, 700, 128, 4, "bf16", 0, 0),
    (5, 129, 64, 28, 4, "bf16", 8, 0),
    (5, 129, 500, 28, 4, "bf16", 8, 0),  # the same behind a walk long enough for 16 x 16 MFMAs
])
@pytest.mark.parametrize("spread", [0, 1])
def test_int8_cache(xh, orc, B, S, past, qh, kvh, kind, extra, skip, spread):
    """spread: the values' sizes go up and down by powers of ten from token to token and block to block, so that the scale they are taken relative to moves."""
    assert xh.attention_prefill_form(qh, kvh, B, S, past, int8=True) == (2 if past + S // 2 >= 256 else 1)
    rng = np.random.default_rng(S * 37 + past)
    n = past + S
    k, v = (rng.standard_normal((B, n, kvh * D)).astype(np.float32) for _ in range(2))
    if spread:
        v *= (10.0 ** (-rng.integers(0, 3, n) - 2.0 * ((np.arange(n) // 48) % 3)))[None, :, None].astype(np.float32)
        v[:, n // 2] *= 1e3
    kc, vc, dc = _cache(xh, orc, k, v, 1)
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)))
    got = _attend(xh, orc, dc, q, B, S, qh, past, xh.BF16 if kind == "bf16" else xh.F32, qh * D + extra, skip)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, [past] * B, SCALE)
    # fp16 products of probabilities and scales: 2^-11 of a value each, or 2^-25 of the largest that the 32 columns of the query's wave see; bf16 results 2^-9 on top
    vf = vc.as_f32()
    size = orc.attention_ref_f64(q, kc.as_f32(), np.abs(vf), qh, kvh, D, [S] * B, [past] * B, SCALE)
    largest = np.maximum.accumulate(np.abs(vf).max(3), 2)  # [B, KV heads, tokens]
    column = np.arange(S)[:, None] * (qh // kvh) + np.arange(qh // kvh)
    seen = past + np.minimum(column // 32 * 32 + 31, S * (qh // kvh) - 1) // (qh // kvh)
    largest = largest[:, :, seen].transpose(0, 2, 1, 3).reshape(B * S, qh, 1).repeat(D, 2).reshape(size.shape)
    bound = 2.0 ** -11 * size + 2.0 ** -25 * n * largest + 2.0 ** -18 * size + np.abs(ref) * (2.0 ** -8 if kind == "bf16" else 0.0)
    assert (np.abs(got - ref) <= bound).all(), (np.abs(got - ref) / bound).max()
    # and no query's row is noise: but for those that see a token a thousand times as large in their wave
    near = bound.reshape(B * S, qh, D).max(2) < 0.1 * np.abs(ref).reshape(B * S, qh, D).max(2)
    assert near.mean() > 0.8, near.mean()
    dc.free()


@pytest.mark.parametrize("kind", ["fp16", "int8"])
@pytest.mark.parametrize("drop", [12.0, 15.5, 18.0, 21.0])
def test_weights_among_the_subnormal_values(xh, orc, kind, drop):
    """One key far above all others, whose probabilities lie at 2^-drop of its own: subnormal in fp16 from 2^-14 on.  Thousands of them are a share of the
    result all the same, above and below the line alike."""
    S, qh, kvh, int8 = 3000, 32, 8, int(kind == "int8")
    rng = np.random.default_rng(int(drop))
    k, v = np.zeros((1, S, kvh * D), np.float32), 1.0 + rng.standard_normal((1, S, kvh * D)).astype(np.float32)
    k.reshape(S, kvh, D)[0, :, 0] = drop * np.log(2.0) / SCALE / 2.0
    k.reshape(S, kvh, D)[1:, :, 1] = 0.05 * rng.standard_normal((S - 1, kvh))
    v[0, 0] = 4.0  # (a share lost above or below the line moves the result by as much times the distance of 3 from the others' mean)
    kc, vc, dc = _cache(xh, orc, k, v, int8)
    q = orc.round_bf16(np.tile(np.eye(1, D, 0) * 2.0 + np.eye(1, D, 1), (S, qh)))
    got = _attend(xh, orc, dc, q, 1, S, qh, 0, xh.F32, qh * D, 0).reshape(S, qh, D)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S], [0], SCALE).reshape(S, qh, D)
    # a probability in fp16 is off by 2^-11 of itself or 2^-25 at most (INT8: its product with a value scale relative to the one in use, the first key's 1.0
    # among them), times a value's distance from the result, of up to 8; fp32 sums 2^-18 on top
    n = np.arange(1, S + 1)[:, None, None]
    size = 8.0 * (2.0 ** -11 * np.minimum(n * 2.0 ** -drop, 1.0) + 2.0 ** -25 * n) + (4.0 * 2.0 ** -11 if int8 else 0.0) + 8.0 * 2.0 ** -18
    assert (np.abs(got - ref) <= size).all(), (np.abs(got - ref) / size).max()
    dc.free()


@pytest.mark.parametrize("scale", [-0.3, 0.0, 1e-30, 1.5e-6, 3e-4, 0.04, 0.11, 0.3, 0.99, 3.0])
@pytest.mark.parametrize("size", [0.05, 1.0, 1e4])
@pytest.mark.parametrize("kind", ["fp16", "int8"])
def test_any_softmax_scale(xh, orc, scale, size, kind):
    """Scales of any size and sign, with queries and keys such that the scores are about one (or, where they can't be, smaller): no query loses bits."""
    B, S, qh, kvh = 20, 64, 32, 8
    rng = np.random.default_rng(int(abs(scale) * 1e6) % 1000 + int(size))
    key = min(0.1 / max(abs(scale) * size, 1e-12), 8e3)
    k, v = (rng.standard_normal((B, S, kvh * D)).astype(np.float32) * by for by in (key, 1.0))
    kc, vc, dc = _cache(xh, orc, k, v, int(kind == "int8"))
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)) * size)
    got = _attend(xh, orc, dc, q, B, S, qh, 0, xh.F32, qh * D, 0, scale)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, [0] * B, scale)
    # every probability (INT8: product of probability and scale) in fp16, 2^-11 of it at most and half of that in the root mean square at random; an INT8 cache's
    # value scales beside 1.2 times that; the first tokens, of one value, have nothing to average
    off = np.sqrt(((got - ref) ** 2).reshape(B, S, -1).mean((0, 2))) / np.sqrt((ref ** 2).reshape(B, S, -1).mean((0, 2)))
    assert off.max() < 4e-4, off
    dc.free()


@pytest.mark.parametrize("B,S,past,qh,kvh,kind,extra,skip", [
    (3, 1025, 500, 32, 8, "bf16", 0, 0),  # 33 workgroups a pair, the last of 4 columns
    (5, 515, 1101, 28, 4, "bf16", 8, 8),  # 7 heads a group: a wave's tiles of 16 columns begin inside a token; 21 columns in the last workgroup
    (2, 301, 2003, 128, 2, "f32", 4, 0),  # 64 heads a group: both tiles of a wave belong to one token
    (8, 1025, 800, 8, 8, "bf16", 1, 1),  # one head a group: every column another token; rows on 2-byte borders
    (8, 129, 1233, 64, 8, "bf16", 4, 4),
])
@pytest.mark.parametrize("score,scale", [(None, SCALE), (-1e30, SCALE), (3000.0, SCALE), (None, 1e-4)])
def test_launches_that_fill_the_device(xh, orc, B, S, past, qh, kvh, kind, extra, skip, score, scale):
    """Enough workgroups and (workgroup, 32-token block) pairs for the form in 16 x 16 MFMAs.  The first 40 tokens score as the others,
    minus infinity, or so high that the others' weights vanish."""
    rng = np.random.default_rng(S * 31 + past)
    assert xh.attention_prefill_form(qh, kvh, B, S, past) == 2
    k, v = (rng.standard_normal((B, past + S, kvh * D)).astype(np.float32) for _ in range(2))
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)))
    if score is not None:
        k.reshape(B, past + S, kvh, D)[:, :40, :, 0] = score
        k.reshape(B, past + S, kvh, D)[:, 40:, :, 0] = 0.0
        q.reshape(B * S, qh, D)[:, :, 0] = 1.0
    kc, vc, dc = _cache(xh, orc, k, v)
    got = _attend(xh, orc, dc, q, B, S, qh, past, xh.BF16 if kind == "bf16" else xh.F32, qh * D + extra, skip, scale)
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, [past] * B, scale)
    # fp16 probabilities: 2^-11 of a value each; bf16 results 2^-9 on top
    assert (np.abs(got - ref) <= 3e-3 + np.abs(ref) * (2.0 ** -8 if kind == "bf16" else 0.0)).all(), np.abs(got - ref).max()
    dc.free()
