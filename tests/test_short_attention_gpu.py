"""Attention over contexts that one workgroup of eight waves walks: fewer blocks than waves, one each, more; the longest that takes this form and one token
more; positions from the host and from device memory; one query head a KV head, several, several rows."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
D = 128
SCALE = 1.0 / np.sqrt(D)
_streams = []


@pytest.mark.parametrize("kind", ["fp16", "int8"])
@pytest.mark.parametrize("B,S,qh,kvh", [(1, 1, 32, 32), (3, 1, 32, 8), (2, 3, 12, 4), (1, 5, 32, 8)])
@pytest.mark.parametrize("tokens", [129, 160, 256, 257, 320, 321, 384, 385])
def test_short_contexts(kind, B, S, qh, kvh, tokens):
    from oracle import pyoracle as orc
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    code = 1 if kind == "int8" else 0
    rng = np.random.default_rng(tokens * 7 + B + S + code)
    k, v = (rng.standard_normal((B, tokens, kvh * D)).astype(np.float32) for _ in range(2))
    kc, vc = orc.KVCache(code, B, kvh, tokens, D), orc.KVCache(code, B, kvh, tokens, D)
    for b in range(B):
        kc.store(b, 0, k[b])
        vc.store(b, 0, v[b])
    dc = xh.KVCache(xh.INT8 if code else xh.FP16, B, kvh, tokens, D)
    dc.load(0, kc.data, kc.scales)
    dc.load(1, vc.data, vc.scales)
    q = orc.round_bf16(rng.standard_normal((B * S, qh * D)))
    qd = xh.DeviceBuffer.from_numpy(orc.to_bf16(q))
    od = xh.DeviceBuffer.from_numpy(np.zeros(q.shape, np.float32))
    own = [max(tokens - S - 40 * b, 0) for b in range(B)]  # some sequences end blocks earlier
    pd = xh.DeviceBuffer.from_numpy(np.array(own, np.int32))
    for call in (xh.attention, xh.attention_static):
        for past, at in (([tokens - S] * B, None), (own, pd.ptr)):
            call(dc, qd.ptr, q.shape[1], od.ptr, q.shape[1], xh.F32, B, S, qh, SCALE, tokens - S, at)
            xh.synchronize()
            got = od.to_numpy(np.float32, q.shape)
            ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [S] * B, past, SCALE)
            # probabilities (and, of an INT8 cache, their products with the values' scales) in fp16: 2^-11 of a value each
            assert np.abs(got - ref).max() < 3e-3, (call.__name__, past)
    dc.free()


@pytest.mark.parametrize("kind", ["fp16", "int8"])
def test_longer_call_captured_behind_a_short_one(kind):
    """A stream's first call brings the workspace of split contexts: one that does not need it, then, captured, one that does."""
    from oracle import pyoracle as orc
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    code, qh, kvh, tokens = int(kind == "int8"), 32, 8, 1000
    rng = np.random.default_rng(91 + code)
    kc, vc = orc.KVCache(code, 1, kvh, tokens, D), orc.KVCache(code, 1, kvh, tokens, D)
    kc.store(0, 0, rng.standard_normal((tokens, kvh * D)).astype(np.float32))
    vc.store(0, 0, rng.standard_normal((tokens, kvh * D)).astype(np.float32))
    dc = xh.KVCache(xh.INT8 if code else xh.FP16, 1, kvh, tokens, D)
    dc.load(0, kc.data, kc.scales)
    dc.load(1, vc.data, vc.scales)
    q = orc.round_bf16(rng.standard_normal((1, qh * D)))
    qd, od = xh.DeviceBuffer.from_numpy(orc.to_bf16(q)), xh.DeviceBuffer(q.size * 4)
    stream = xh.Stream()
    _streams.append(stream)  # (a stream gone leaves its handle, and with it its workspace, to the next)

    def call(past):
        xh.attention(dc, qd.ptr, qh * D, od.ptr, qh * D, xh.F32, 1, 1, qh, SCALE, past, None, stream.h)

    call(199)
    stream.synchronize()
    xh.check(xh.lib.xfthip_graph_begin(stream.h))
    call(tokens - 1)
    g = C.c_void_p()
    xh.check(xh.lib.xfthip_graph_end(stream.h, C.byref(g)))
    ref = orc.attention_ref_f64(q, kc.as_f32(), vc.as_f32(), qh, kvh, D, [1], [tokens - 1], SCALE)
    for _ in range(3):
        od.zero()
        xh.synchronize()
        xh.check(xh.lib.xfthip_graph_launch(g, stream.h))
        stream.synchronize()
        assert np.abs(od.to_numpy(np.float32, q.shape) - ref).max() < 3e-3
    xh.check(xh.lib.xfthip_graph_destroy(g))
    dc.free()
