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
