"""The delta rule's scan with one and with two columns a group of lanes, full chunks of tokens and remainders, states that go on from a step before;
one decay a key channel and one a head."""
import numpy as np
import pytest

import duvadra_util as one_decay
import plan_util as many_decays
from oracle import duvadra_ref, pinepel_ref

pytestmark = pytest.mark.gpu

# tokens of every segment in the first and in the second step: chunks of 8 and what is left of them, beside segments that begin or end early
FIRST, SECOND = [1, 8, 17, 33, 7, 16, 64, 2], [40, 9, 1, 8, 25, 3, 16, 7]


# (key width, value width, heads.  8 segments of the first three and of the fourth take two columns a group of lanes on 256 compute units, the others one)
@pytest.mark.parametrize("dim,vdim,heads", [(128, 128, 16), (64, 64, 64), (200, 48, 32), (128, 96, 22), (128, 128, 3), (32, 64, 8)])
@pytest.mark.parametrize("decay", ["channel", "head"])
def test_scan(dim, vdim, heads, decay):
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    kv = heads // 2 if heads % 2 == 0 else heads
    if decay == "channel":
        u, ref = many_decays, pinepel_ref
        cfg = u.config([u.delta(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, conv=4)])
    else:
        u, ref = one_decay, duvadra_ref
        cfg = u.config([(u.windowed_delta(r_heads=heads, r_kv_heads=kv, r_dim=dim, r_vdim=vdim, left=0.0), None)])
    bits = u.weights(cfg, 21)
    case = u.Case(xh, u.build_plan(xh, cfg, bits), u.oracle_weights(bits), lambda w, t: ref.forward(cfg, w, t), "f32", 3e-5, 8, 128, 256)
    rng = np.random.default_rng(dim + heads)
    texts = [rng.integers(0, cfg["vocab"], a + b) for a, b in zip(FIRST, SECOND)]
    want = [case.want(t) for t in texts]
    for ends, begins, what in ((FIRST, [0] * 8, "first step"), ([len(t) for t in texts], FIRST, "second step")):
        got = case.model.step([(i, t[b:e], list(range(e - b))) for i, (t, b, e) in enumerate(zip(texts, begins, ends))])
        case.check(got, np.concatenate([w[b:e] for w, b, e in zip(want, begins, ends)]), what)
    case.free()


# Segments 16 tokens at a time: a token beside it and less, whole chunks, one of a single token, several pairs and an odd one of them, single tokens of other sequences beside them
LONG, THEN = [1, 16, 17, 140, 15, 32, 47, 129], [130, 9, 33, 1, 16, 3, 31, 48]


# (one tile of 16 columns a wave and, from 1024 tiles on 256 compute units, two; key widths of 64, 128 and 256)
@pytest.mark.parametrize("dim,vdim,heads,few", [(128, 128, 16, 0), (128, 96, 4, 0), (64, 64, 4, 0), (50, 64, 64, 0), (200, 96, 6, 0), (256, 64, 32, 0), (128, 64, 2, 3)])
@pytest.mark.parametrize("decay", ["channel", "head"])
def test_scan_in_chunks(dim, vdim, heads, few, decay):
    """few: that many of the sequences, beginning with the longest"""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    kv = heads // 2
    if decay == "channel":
        u, ref = many_decays, pinepel_ref
        cfg = u.config([u.delta(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, conv=4)])
    else:
        u, ref = one_decay, duvadra_ref
        cfg = u.config([(u.windowed_delta(r_heads=heads, r_kv_heads=kv, r_dim=dim, r_vdim=vdim, left=0.0), None)])
    bits = u.weights(cfg, 22)
    case = u.Case(xh, u.build_plan(xh, cfg, bits), u.oracle_weights(bits), lambda w, t: ref.forward(cfg, w, t), "f32", 3e-5, 8, 384, 512)
    rng = np.random.default_rng(dim + heads)
    first, then = (LONG[3:3 + few], THEN[3:3 + few]) if few else (LONG, THEN)
    texts = [rng.integers(0, cfg["vocab"], a + b) for a, b in zip(first, then)]
    want = [case.want(t) for t in texts]
    for ends, begins, what in ((first, [0] * 8, "first step"), ([len(t) for t in texts], first, "second step")):
        got = case.model.step([(i, t[b:e], list(range(e - b))) for i, (t, b, e) in enumerate(zip(texts, begins, ends))])
        case.check(got, np.concatenate([w[b:e] for w, b, e in zip(want, begins, ends)]), what)
    case.free()


@pytest.mark.parametrize("at", [0, 7, 16, 37])
@pytest.mark.parametrize("what", [0x7FC0, 0x7F80, 0xFF80])  # NaN, infinities
def test_chunks_and_what_is_not_finite(at, what):
    """A token of which nothing is finite: the tokens in front of it, in its chunk too, are as they are without it, those behind it are lost as they are token by token."""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    u, ref = many_decays, pinepel_ref
    cfg = u.config([u.delta(heads=4, kv_heads=2, dim=128, vdim=64, conv=4)])
    bits = u.weights(cfg, 23)
    sound = u.oracle_weights(bits)
    bits["embed"][5, 3] = what
    case = u.Case(xh, u.build_plan(xh, cfg, bits), sound, lambda w, t: ref.forward(cfg, w, t), "f32", 3e-5, 8, 384, 512)
    rng = np.random.default_rng(at)
    texts = [rng.integers(6, cfg["vocab"], 45) for _ in range(2)]
    want = [case.want(t) for t in texts]
    texts[0][at] = 5
    got = case.model.step([(i, t, list(range(45))) for i, t in enumerate(texts)])
    assert not np.isfinite(got[at:45]).any()
    case.check(np.concatenate([got[:at], got[45:]]), np.concatenate([want[0][:at], want[1]]), "the others")
    case.free()
