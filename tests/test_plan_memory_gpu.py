"""A device that is short of memory: a plan model that has room for one context in the expanded form of latent attention, but not for all of a step's; a step
without a buffer for the parts of a product whose K is split."""
import ctypes as C

import numpy as np
import pytest

import duvadra_util
import plan_util as u
from oracle import pinepel_ref as ref

pytestmark = pytest.mark.gpu
HEADS, DIM, ROT, RANK, SLOTS, SEQ, TOKENS = 64, 128, 64, 128, 256, 64, 16384


def left():
    from xfastertransformer_amd import capi as xh
    free, device = C.c_size_t(), C.c_size_t()
    assert xh.lib.hipMemGetInfo(C.byref(free), C.byref(device)) == 0  # (of the runtime that the library is linked with)
    return free.value


def test_refused_allocation_is_told_once():
    """the call behind one that found no memory runs"""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    x, w, out = xh.DeviceBuffer.from_numpy(np.arange(256, dtype=np.float32)), xh.DeviceBuffer.from_numpy(np.ones(256, np.float32)), xh.DeviceBuffer(1024)
    with pytest.raises(xh.XftHipError, match="memory"):
        xh.DeviceBuffer(1 << 50)
    xh.rmsnorm(out.ptr, xh.F32, x.ptr, xh.F32, w.ptr, 1, 256)
    y = np.arange(256.0)
    np.testing.assert_allclose(out.to_numpy(np.float32, 256), y / np.sqrt((y * y).mean() + 1e-6), rtol=1e-6)


def test_model_that_just_fits():
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    cfg = u.config([u.latent(heads=HEADS, dim=DIM, rot=ROT, vdim=DIM, kv_rank=RANK, q_rank=64)])
    bits = u.weights(cfg, 17)
    plan, w = u.build_plan(xh, cfg, bits), u.oracle_weights(bits)
    rng = np.random.default_rng(4)
    texts = [rng.integers(0, cfg["vocab"], int(n)) for n in rng.integers(33, SEQ + 1, 40)]
    want = np.stack([ref.forward(cfg, w, t)[-1] for t in texts])

    def step(model):
        got = model.step([(i, t, [len(t) - 1]) for i, t in enumerate(texts)])
        assert u.rel_rms(got, want).max() < 0.06

    before = left()
    model = xh.PlanModel(plan, xh.BF16, SLOTS, SEQ, TOKENS)
    used = before - left()
    step(model)  # (and the stream has its scratch memory)
    model.free()
    more = (TOKENS + 31 * 32 - SEQ - 32) * (2 * HEADS * DIM + RANK + ROT) * 2  # the contexts behind the first
    assert 0.2 * used < more < 0.8 * used
    room, ballast = used - more // 2, []
    while left() > room + (64 << 20):
        ballast.append(xh.DeviceBuffer(min(left() - room, 16 << 30)))
    model = xh.PlanModel(plan, xh.BF16, SLOTS, SEQ, TOKENS)
    step(model)
    model.free()
    for b in ballast:
        b.free()
    plan.free()


def test_step_that_finds_no_memory():
    """A step of one token a sequence that fails half way, for want of a buffer for a product's parts on a stream of its own, leaves the sequences where they
    stood: the same step, repeated, finds their positions and the tokens before (the pair embedding reads them) as they were."""
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    n, parts = 40, 64 << 20  # (a product of 40 rows, 4096 deep, takes its K in parts)
    cfg = duvadra_util.config([(duvadra_util.chunked(), duvadra_util.dense(ff=4096))])
    plan = duvadra_util.build_plan(xh, cfg, duvadra_util.weights(cfg, 8))
    model, twin = (xh.PlanModel(plan, xh.BF16, n, 64, n) for _ in range(2))
    rng, streams = np.random.default_rng(2), [xh.Stream() for _ in range(4)]
    draw = lambda: rng.integers(0, cfg["vocab"], n).astype(np.int32)
    entries = lambda tokens: [(i, tokens[i:i + 1], [0]) for i in range(len(tokens))]
    tokens = draw()
    assert np.array_equal(model.step(entries(tokens)), twin.step(entries(tokens)))
    for s in streams:  # (one token: no parts; what a stream needs otherwise it has then)
        few = draw()[:1]
        assert np.array_equal(model.step(entries(few), s.h), twin.step(entries(few)))
    ballast = []
    while left() > parts - (8 << 20):
        ballast.append(xh.DeviceBuffer(min(left() - (parts - (32 << 20)), 16 << 30)))
    failed = 0
    for s in streams:  # (a stream may have the handle, and the buffer, of one that is gone)
        tokens = draw()
        want = twin.step(entries(tokens))
        try:
            got = model.step(entries(tokens), s.h)
        except xh.XftHipError:
            failed += 1
            break
        assert np.array_equal(got, want)
    for b in ballast:
        b.free()
    assert failed
    assert np.array_equal(model.step(entries(tokens), s.h), want)
    tokens = draw()
    assert np.array_equal(model.step(entries(tokens), s.h), twin.step(entries(tokens)))
    model.free()
    twin.free()
    plan.free()
