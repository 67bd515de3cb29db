"""A plan model's logits on their way to the host: pieces and their borders, vocabularies whose rows begin anywhere, more rows than go at a time."""
import numpy as np
import pytest

import plan_util as u
from oracle import pinepel_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,tokens", [(1003, 1), (1003, 33), (4097, 8), (33001, 1), (33001, 8), (65537, 5)])
def test_logits_of_all_sizes(vocab, tokens):
    """1 to 8 pieces, full and partly filled, on 16-byte borders and off them: the last piece of 33001 values holds 233, of 4097 x 8 eight."""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    cfg = u.config([u.latent()], vocab=vocab)
    bits = u.weights(cfg, 5)
    w = u.oracle_weights(bits)
    model = xh.PlanModel(u.build_plan(xh, cfg, bits), xh.F32, 2, 64, 64)
    ids = np.random.default_rng(vocab + tokens).integers(0, vocab, tokens)
    want = ref.forward(cfg, w, ids)
    for _ in range(3):  # (the flags and counts of the copy before stay behind)
        got = model.step([(0, ids, list(range(tokens)))])
        assert u.rel_rms(got, want).max() < 3e-5 and np.abs(got - want).max() < 1e-3 * want.std()
        one = model.step([(1, ids[:1], [0])])
        assert u.rel_rms(one, want[:1]).max() < 3e-5
        model.seq_release(0)
        model.seq_release(1)
    model.free()
