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


def _attend(xh, orc, dc, q, B, S, qh, past, out_dtype, pitch, skip):
    """Results at `skip` elements from a 256-byte border, rows `pitch` elements apart; what lies between the rows stays as it is."""
    rows, width, bf16 = q.shape[0], q.shape[1], out_dtype == xh.BF16
    qd = xh.DeviceBuffer.from_numpy(orc.to_bf16(q))
    mark = np.full(rows * pitch + skip, 7.0, np.float32)
    od = xh.DeviceBuffer.from_numpy(orc.to_bf16(mark) if bf16 else mark)
    at = C.c_void_p(od.ptr.value + skip * (2 if bf16 else 4))
    xh.attention(dc, qd.ptr, width, at, pitch, out_dtype, B, S, qh, SCALE, past)
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
    (40, 2, 700, 32, 1, "bf16", 0, 0),  # a token's heads fill a wave; the first three blocks lie before all new tokens
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
    (40, 2, 700, 32, 1, "bf16", 0, 0),
    (5, 129, 64, 28, 4, "bf16", 8, 0),
])
@pytest.mark.parametrize("spread", [0, 1])
def test_int8_cache(xh, orc, B, S, past, qh, kvh, kind, extra, skip, spread):
    """spread: the values' sizes go up and down by powers of ten from token to token and block to block, so that the scale they are taken relative to moves."""
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
    # fp16 products of probabilities and scales: 2^-11 of a value each, or 2^-25 of 2^8 times the largest scale's; bf16 results 2^-9 on top
    size = np.abs(vc.as_f32()).max()
    assert (np.abs(got - ref) <= 6e-4 * max(size, 1.0) + 3e-3 + np.abs(ref) * (2.0 ** -8 if kind == "bf16" else 0.0)).all(), np.abs(got - ref).max()
    dc.free()
