"""The delta rule token by token, with one and with two columns a group of lanes, full chunks of tokens and remainders, states that go on from a step before, and 16
tokens at a time; one decay a key channel and one a head."""
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
    assert not case.model.delta_chunks(False)  # token by token, whatever the lengths
    rng = np.random.default_rng(dim + heads)
    texts = [rng.integers(0, cfg["vocab"], a + b) for a, b in zip(FIRST, SECOND)]
    want = [case.want(t) for t in texts]
    for ends, begins, what in ((FIRST, [0] * 8, "first step"), ([len(t) for t in texts], FIRST, "second step")):
        got = case.model.step([(i, t[b:e], list(range(e - b))) for i, (t, b, e) in enumerate(zip(texts, begins, ends))])
        case.check(got, np.concatenate([w[b:e] for w, b, e in zip(want, begins, ends)]), what)
    case.free()


# Segments 16 tokens at a time: a token beside it and less, whole chunks, one of a single token, several pairs and an odd one of them, single tokens of other sequences beside them
LONG, THEN = [1, 16, 17, 140, 15, 32, 47, 129], [130, 9, 33, 1, 16, 3, 31, 48]


def held(dim, vdim, heads, decay, steps, forms, tokens=512):
    """A layer over several steps.  steps: the tokens of every sequence, step by step; forms: what xh.delta_forms has to say of each of them"""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    kv = heads // 2
    if decay == "channel":
        u, ref = many_decays, pinepel_ref
        cfg = u.config([u.delta(heads=heads, kv_heads=kv, dim=dim, vdim=vdim, conv=4)])
    else:
        u, ref = one_decay, duvadra_ref
        cfg = u.config([(u.windowed_delta(r_heads=heads, r_kv_heads=kv, r_dim=dim, r_vdim=vdim, left=0.0), None)])
    for lens, form in zip(steps, forms):
        assert set(xh.delta_forms(heads, dim, vdim, 4, decay == "head", lens)) == form
    bits = u.weights(cfg, 22)
    n = len(steps[0])
    case = u.Case(xh, u.build_plan(xh, cfg, bits), u.oracle_weights(bits), lambda w, t: ref.forward(cfg, w, t), "f32", 3e-5, n, 384, tokens, n * 384)
    assert case.model.delta_chunks()
    rng = np.random.default_rng(dim + heads)
    ends = np.cumsum([[0] * n] + [list(s) for s in steps], 0)
    texts = [rng.integers(0, cfg["vocab"], e) for e in ends[-1]]
    want = [case.want(t) for t in texts]
    for k in range(len(steps)):
        part = list(zip(ends[k], ends[k + 1]))
        got = case.model.step([(i, t[b:e], list(range(e - b))) for i, (t, (b, e)) in enumerate(zip(texts, part))])
        case.check(got, np.concatenate([w[b:e] for w, (b, e) in zip(want, part)]), f"step {k}")
    case.free()


# (one tile of 16 columns a wave; key widths of 64, 128 and 256.  1024 tiles on 256 compute units are enough for each segment to go by its own length: those of 64 tokens and more
# (128 with one decay a head) in chunks, the others token by token; the last case's values are too wide for the preparation that walks several tokens.)
@pytest.mark.parametrize("dim,vdim,heads,few,forms", [(128, 128, 16, 0, {0, 1}), (128, 96, 4, 0, {1}), (64, 64, 4, 0, {1}), (50, 64, 64, 0, {0, 1}), (200, 96, 6, 0, {1}), (256, 64, 32, 0, {0, 1}), (128, 64, 2, 3, {1}),
                                                     (64, 288, 8, 0, {0, 1})])
@pytest.mark.parametrize("decay", ["channel", "head"])
def test_scan_in_chunks(dim, vdim, heads, few, forms, decay):
    """few: that many of the sequences, beginning with the longest"""
    first, then = (LONG[3:3 + few], THEN[3:3 + few]) if few else (LONG, THEN)
    held(dim, vdim, heads, decay, [first, then], [forms, forms])


# (two tiles of 16 columns a wave; a few short segments go with the long ones)
@pytest.mark.parametrize("dim,vdim,heads", [(128, 128, 16), (50, 64, 64), (256, 64, 32)])
@pytest.mark.parametrize("decay", ["channel", "head"])
def test_scan_in_chunks_two_tiles(dim, vdim, heads, decay):
    held(dim, vdim, heads, decay, [[140, 129, 128, 131, 144, 150, 160, 133, 5], [129, 130, 145, 128, 160, 133, 131, 150, 1]], [{1}, {1}], 1200)


@pytest.mark.parametrize("dim,vdim,heads", [(128, 128, 16), (64, 64, 32), (256, 64, 32)])
@pytest.mark.parametrize("decay", ["channel", "head"])
def test_prompts_beside_decoding_sequences(dim, vdim, heads, decay):
    """Single tokens by the kernel for them beside prompts in chunks, which go on one token at a time while the next prompt comes."""
    held(dim, vdim, heads, decay, [[3, 2, 1, 4, 5, 1, 2, 2, 130, 3], [1, 1, 140, 1, 1, 1, 1, 1, 1, 129], [1] * 10, [1, 130, 1, 1, 1, 1, 1, 1, 17, 1]], [{0, 1}, {0, 1}, {0}, {0, 1}])


def test_more_segments_than_a_launch_names():
    lens = [32 + i % 5 for i in range(131)]
    held(64, 32, 4, "channel", [lens, lens[::-1]], [{1}, {1}], 4608)


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
    assert case.model.delta_chunks() and xh.delta_forms(4, 128, 64, 4, False, [45, 45]) == [1, 1]
    rng = np.random.default_rng(at)
    texts = [rng.integers(6, cfg["vocab"], 45) for _ in range(2)]
    want = [case.want(t) for t in texts]
    texts[0][at] = 5
    got = case.model.step([(i, t, list(range(45))) for i, t in enumerate(texts)])
    assert not np.isfinite(got[at:45]).any()
    case.check(np.concatenate([got[:at], got[45:]]), np.concatenate([want[0][:at], want[1]]), "the others")
    case.free()


def test_records_given_back_and_held_again():
    """A sequence that goes on in the other form from step to step, and back."""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    u, ref = many_decays, pinepel_ref
    cfg = u.config([u.delta(heads=4, kv_heads=2, dim=100, vdim=64, conv=3)])
    bits = u.weights(cfg, 24)
    case = u.Case(xh, u.build_plan(xh, cfg, bits), u.oracle_weights(bits), lambda w, t: ref.forward(cfg, w, t), "f32", 3e-5, 2, 384, 256)
    text = np.random.default_rng(5).integers(0, cfg["vocab"], 200)
    want, at = case.want(text), 0
    for use, n in ((None, 40), (False, 35), (False, 20), (True, 33), (True, 50), (False, 1), (True, 21)):
        assert case.model.delta_chunks(use) == (use is not False) == case.model.delta_chunks()
        case.check(case.model.step([(1, text[at:at + n], list(range(n)))]), want[at:at + n], f"at {at}")
        at += n
    case.free()


def test_models_without_such_layers_hold_none():
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    u = many_decays
    cfg = u.config([u.delta(heads=2, kv_heads=2, dim=32, vdim=32, conv=4)])  # (keys too narrow)
    plan = u.build_plan(xh, cfg, u.weights(cfg, 25))
    model = xh.PlanModel(plan, xh.F32, 2, 64, 64)
    assert not model.delta_chunks() and not model.delta_chunks(True) and not model.delta_chunks(False)
    model.free()
    plan.free()
