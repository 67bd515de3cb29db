"""Latent attention's expanded form over several long segments of one step: one gather, one pair of products and one launch a group of them."""
import numpy as np
import pytest

import plan_util as u
from oracle import pinepel_ref as ref

pytestmark = pytest.mark.gpu


def steps(case, sequences, cuts):
    """sequence i in portions that end at cuts[k][i]; all logits of every step checked"""
    want = [case.want(t) for t in sequences]
    at = [0] * len(sequences)
    for k, ends in enumerate(cuts):
        entries = [(i, t[at[i]:e], list(range(e - at[i]))) for i, (t, e) in enumerate(zip(sequences, ends)) if e > at[i]]
        case.check(case.model.step(entries), np.concatenate([want[i][at[i]:e] for i, e in enumerate(ends) if e > at[i]]), f"step {k}")
        at = list(ends)


def case_of(layers, slots, max_seq, max_tokens):
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    cfg = u.config(layers)
    bits = u.weights(cfg, 11)
    return cfg, u.Case(xh, u.build_plan(xh, cfg, bits), u.oracle_weights(bits), lambda w, t: ref.forward(cfg, w, t), "bf16", 0.06, slots, max_seq, max_tokens)


@pytest.mark.parametrize("window", [None, 50])
def test_portions_of_unequal_segments(window):
    """Short and long segments in turn, ends on and off blocks of 32, contexts that begin at a window's edge; the second step's contexts are longer
    together than the buffers, so that they go in groups."""
    first, second = [33, 1, 128, 250, 31, 64, 129, 40], [97, 2, 160, 300, 200, 96, 290, 75]
    cfg, c = case_of([u.latent(window=window), u.latent()], 8, 320, 720)
    rng = np.random.default_rng(2)
    steps(c, [rng.integers(0, cfg["vocab"], n) for n in second], [first, second])
    c.free()


def test_more_segments_than_a_group():
    cfg, c = case_of([u.latent()], 70, 64, 70 * 40)
    rng = np.random.default_rng(3)
    lengths = [int(n) for n in rng.integers(32, 41, 70)]
    steps(c, [rng.integers(0, cfg["vocab"], n) for n in lengths], [lengths])
    c.free()


@pytest.mark.parametrize("tokens,heads,kv_rank,batch", [(n, 3, 512, 1) for n in (40, 200, 400, 700, 1300, 2500)] + [(n, 40, 40, 2) for n in (40, 200, 700)])
def test_splits_of_a_context(tokens, heads, kv_rank, batch):
    """One new token behind contexts of 2 to 64 splits: each number of thread groups that share them in the merge, one column group and two."""
    cfg, c = case_of([u.latent(heads=heads, kv_rank=kv_rank)], batch, 2560, batch * tokens)
    rng = np.random.default_rng(tokens)
    lengths = [tokens - 31 * i // 2 for i in range(batch)]
    steps(c, [rng.integers(0, cfg["vocab"], n + 1) for n in lengths], [lengths, [n + 1 for n in lengths]])
    c.free()
