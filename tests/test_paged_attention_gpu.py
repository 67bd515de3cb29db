"""Attention over a block-paged BF16 KV cache (xft::invokeAttention, include/layers_attention.h:22-59,
src/kernels/attention_kernels.cpp:24-157) on the GPU against the CPU oracle: decode over ragged
contexts through shuffled block tables (MHA and grouped heads, several block sizes, strided rows),
prefill of ragged sequences, and the host entry point driven as a serving loop would drive it
(prefill, then decode steps that grow the tables).  The reference has no test of this function; the
oracle is pinned against float64 brute force in tests/test_oracle_pins.py.
Tolerance: outputs are bf16 (relative step 2^-8); |d| <= 2e-2 and cosine >= 0.9999 on N(0,1) inputs."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def xh():
    from xfastertransformer_amd import capi
    capi.init()
    return capi


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _cos(a, b):
    a, b = a.astype(np.float64).ravel(), b.astype(np.float64).ravel()
    return float(a @ b / np.sqrt((a @ a) * (b @ b)))


def _bf(orc, rng, shape):
    return orc.round_bf16(rng.standard_normal(shape).astype(np.float32))


def _tables(rng, ctx, block_size, block_num, extra=1):
    """Disjoint random blocks for every sequence, enough for ctx[b] + extra tokens."""
    need = [(c + extra + block_size - 1) // block_size for c in ctx]
    assert sum(need) <= block_num
    perm = rng.permutation(block_num)
    tab = np.zeros((len(ctx), max(need)), np.int32)
    at = 0
    for b, n in enumerate(need):
        tab[b, :n] = perm[at:at + n]
        at += n
    return tab, np.asarray(need, np.int32)


@pytest.mark.parametrize("B,qH,kvH,block_size,max_ctx", [(1, 32, 32, 4, 700), (5, 32, 8, 16, 3000), (32, 32, 32, 16, 300),
                                                       (3, 8, 2, 1, 40), (2, 32, 8, 64, 9000)])
def test_paged_decode_matches_oracle(xh, orc, B, qH, kvH, block_size, max_ctx):
    D = 128
    rng = np.random.default_rng(B * 1000 + block_size)
    ctx = rng.integers(0, max_ctx, B).astype(np.int32)
    ctx[0] = max_ctx - 1
    if B > 1:
        ctx[1] = 0  # a sequence whose only token is the new one
    if B > 2:
        ctx[2] = (ctx[2] // block_size) * block_size  # the new token opens a block
    block_num = int(sum((c + 1 + block_size - 1) // block_size for c in ctx)) + 3
    tab, _ = _tables(rng, ctx, block_size, block_num)
    slots = np.asarray([tab[b, ctx[b] // block_size] * block_size + ctx[b] % block_size for b in range(B)], np.int32)
    kc, vc = _bf(orc, rng, (block_num, block_size, kvH, D)), _bf(orc, rng, (block_num, block_size, kvH, D))
    q_stride, kv_stride = qH * D + 64, kvH * D + 8
    q, k, v = _bf(orc, rng, (B, q_stride)), _bf(orc, rng, (B, kv_stride)), _bf(orc, rng, (B, kv_stride))
    dev = lambda a: xh.DeviceBuffer.from_numpy(np.ascontiguousarray(a))
    dkc, dvc = dev(orc.to_bf16(kc)), dev(orc.to_bf16(vc))
    dq, dk, dv = dev(orc.to_bf16(q)), dev(orc.to_bf16(k)), dev(orc.to_bf16(v))
    dt, dc, ds = dev(tab), dev(ctx), dev(slots)
    out = xh.DeviceBuffer(B * qH * D * 2)
    scale = 1.0 / np.sqrt(D)
    xh.paged_attention_decode(out.ptr, dq.ptr, dk.ptr, dv.ptr, qH, kvH, D, q_stride, kv_stride, qH * D, scale, B, dkc.ptr, dvc.ptr,
                              block_num, block_size, dt.ptr, tab.shape[1], dc.ptr, ds.ptr, int(ctx.max()))
    xh.synchronize()
    got = orc.from_bf16(out.to_numpy(np.uint16, (B, qH, D)))
    ref = orc.paged_attention_decode(q[:, :qH * D].reshape(B, qH, D), k[:, :kvH * D].reshape(B, kvH, D),
                                     v[:, :kvH * D].reshape(B, kvH, D), kc, vc, tab, ctx, slots, scale)
    # the new rows reached their slots, nothing else moved (kc / vc were updated in place by the oracle)
    assert np.array_equal(orc.from_bf16(dkc.to_numpy(np.uint16, kc.shape)), kc)
    assert np.array_equal(orc.from_bf16(dvc.to_numpy(np.uint16, vc.shape)), vc)
    err = float(np.abs(got - ref).max())
    print(f"paged decode B={B} heads {qH}/{kvH} block {block_size}: max-abs {err:.2e}, cosine {_cos(got, ref):.6f}", flush=True)
    assert err <= 2e-2 and _cos(got, ref) >= 0.9999


@pytest.mark.parametrize("qH,kvH,lens,block_size", [(32, 32, [7, 128, 300], 16), (32, 8, [1, 1024], 4), (8, 8, [33], 8)])
def test_paged_prefill_matches_oracle(xh, orc, qH, kvH, lens, block_size):
    D = 128
    rng = np.random.default_rng(sum(lens))
    T = sum(lens)
    block_num = sum((L + block_size - 1) // block_size for L in lens) + 2
    tab, _ = _tables(rng, [L - 1 for L in lens], block_size, block_num)
    slots = np.concatenate([[tab[b, t // block_size] * block_size + t % block_size for t in range(L)] for b, L in enumerate(lens)]).astype(np.int32)
    kc, vc = _bf(orc, rng, (block_num, block_size, kvH, D)), _bf(orc, rng, (block_num, block_size, kvH, D))
    q, k, v = _bf(orc, rng, (T, qH, D)), _bf(orc, rng, (T, kvH, D)), _bf(orc, rng, (T, kvH, D))
    dev = lambda a: xh.DeviceBuffer.from_numpy(np.ascontiguousarray(a))
    dkc, dvc = dev(orc.to_bf16(kc)), dev(orc.to_bf16(vc))
    dq, dk, dv, ds = dev(orc.to_bf16(q)), dev(orc.to_bf16(k)), dev(orc.to_bf16(v)), dev(slots)
    out = xh.DeviceBuffer(T * qH * D * 2)
    scale = 1.0 / np.sqrt(D)
    xh.paged_attention_prefill(out.ptr, dq.ptr, dk.ptr, dv.ptr, qH, kvH, D, qH * D, kvH * D, qH * D, scale, lens, dkc.ptr, dvc.ptr,
                               block_num, block_size, ds.ptr)
    xh.synchronize()
    got = orc.from_bf16(out.to_numpy(np.uint16, (T, qH, D)))
    ref = orc.paged_attention_prefill(q, k, v, lens, kc, vc, slots, scale)
    assert np.array_equal(orc.from_bf16(dkc.to_numpy(np.uint16, kc.shape)), kc)
    assert np.array_equal(orc.from_bf16(dvc.to_numpy(np.uint16, vc.shape)), vc)
    err = float(np.abs(got - ref).max())
    print(f"paged prefill heads {qH}/{kvH} lens {lens}: max-abs {err:.2e}, cosine {_cos(got, ref):.6f}", flush=True)
    assert err <= 2e-2 and _cos(got, ref) >= 0.9999


@pytest.mark.parametrize("B,qH,kvH,block_size,max_ctx", [(2, 40, 2, 5, 200), (1, 8, 8, 3, 33), (4, 16, 4, 16, 129), (70, 8, 1, 16, 500), (2, 68, 4, 7, 1500)])
def test_paged_decode_column_groups(xh, orc, B, qH, kvH, block_size, max_ctx):
    """Groups of more than 16 query heads (two column groups, the second of one or four columns), one head a group, block sizes that
    are no power of two, contexts one token past a 32-token block, and enough (sequence, head) pairs for an unsplit context."""
    test_paged_decode_matches_oracle(xh, orc, B, qH, kvH, block_size, max_ctx)


def _decode64(xh, orc, rng, ctx, qH, kvH, change=None, sharp=1.0, block_size=16):
    """A decode call and its softmax in 64 bits: the output, the reference, sum of p |v| and the largest argument of an exponential (in
    magnitude) of every row, sequences in order.  `change(values, tokens in order, sequence)` edits a sequence's values."""
    D, B = 128, len(ctx)
    ctx = np.asarray(ctx, np.int32)
    block_num = int(sum((c + block_size) // block_size for c in ctx)) + 3
    tab, _ = _tables(rng, ctx, block_size, block_num)
    where = [tab[b, np.arange(c + 1) // block_size] * block_size + np.arange(c + 1) % block_size for b, c in enumerate(ctx)]
    kc, vc = _bf(orc, rng, (block_num * block_size, kvH, D)), _bf(orc, rng, (block_num * block_size, kvH, D))
    q = orc.round_bf16(rng.standard_normal((B, qH, D)).astype(np.float32) * sharp)
    if change:
        for b in range(B):
            change(vc, where[b], b)
    slots = np.asarray([w[-1] for w in where], np.int32)
    dev = lambda a: xh.DeviceBuffer.from_numpy(np.ascontiguousarray(a))
    bits = lambda a: dev(orc.to_bf16(a))
    dq, dk, dv, dkc, dvc = bits(q), bits(kc[slots]), bits(vc[slots]), bits(kc), bits(vc)
    dt, dc, ds, out = dev(tab), dev(ctx), dev(slots), xh.DeviceBuffer(B * qH * D * 2)
    xh.paged_attention_decode(out.ptr, dq.ptr, dk.ptr, dv.ptr, qH, kvH, D, qH * D, kvH * D, qH * D, D ** -0.5, B, dkc.ptr, dvc.ptr, block_num,
                              block_size, dt.ptr, tab.shape[1], dc.ptr, ds.ptr, int(ctx.max()))
    xh.synchronize()
    ref, size, slack = (np.zeros((B, qH, D)) for _ in range(3))
    for b in range(B):
        k, v = kc[where[b]].astype(np.float64), vc[where[b]].astype(np.float64)
        for h in range(qH):
            x = k[:, h * kvH // qH] @ q[b, h].astype(np.float64) * D ** -0.5
            p = np.exp(x - x.max())
            p /= p.sum()
            with np.errstate(invalid="ignore"):
                ref[b, h], size[b, h] = p @ v[:, h * kvH // qH], p @ np.abs(v[:, h * kvH // qH])
            # an argument is off by the score's 128 products and additions, and by its own roundings; n probabilities are added up in fp32
            spread = (np.abs(k[:, h * kvH // qH]) @ np.abs(q[b, h].astype(np.float64))).max() * D ** -0.5
            slack[b, h] = 2 * spread * 132 * 2.0 ** -24 + 2 * (np.abs(x).max() + 8) * 2.0 ** -22 + (len(x) + 64) * 2.0 ** -24
    return orc.from_bf16(out.to_numpy(np.uint16, (B, qH, D))).astype(np.float64), ref, size, slack


@pytest.mark.parametrize("qH,kvH,ctx,sharp", [(32, 8, [8200, 33], 1.0), (32, 8, [1500] * 40, 1.0), (8, 1, [4000, 500], 6.0), (4, 4, [3100], 12.0)])
def test_paged_decode_against_64_bits(xh, orc, qH, kvH, ctx, sharp):
    """Bound: half a step of the bf16 result (8 significant bits: 2^-8 of it at most), and what the fp32 scores, exponentials and sums are off by,
    relative to sum p |v|: long contexts whose outputs are small beside the values, and scores of which one takes nearly everything."""
    got, ref, size, slack = _decode64(xh, orc, np.random.default_rng(len(ctx) + qH), ctx, qH, kvH, sharp=sharp)
    bound = np.abs(ref) * 2.0 ** -8 + size * slack
    worst = float((np.abs(got - ref) / bound).max())
    print(f"paged decode heads {qH}/{kvH}, {len(ctx)} x {max(ctx)}, queries x {sharp}: {worst:.3f} of the bound", flush=True)
    assert worst <= 1.0


def test_paged_decode_probabilities_in_32_bits(xh, orc):
    """Values that nearly cancel: the first token's 1 against four tokens of the same lower probability e, whose values are bf16 parts of -1 / e.
    What is left shows the probabilities' own precision.  Bound: an argument of the exponential between -8 and 0, two roundings of it and a unit
    in the last place of the function, 2^-24 of the sums, together below 2^-20 of sum p |v|; a probability in 16 bits is off by up to 2^-17."""
    D, H, rng = 128, 32, np.random.default_rng(2)
    q, k, v = np.zeros((1, H, D), np.float32), np.zeros((5, H, D), np.float32), np.zeros((5, H, D), np.float32)
    q[0, :, 0] = 1.0
    k[1:, :, 0] = orc.round_bf16(-rng.uniform(5, 80, H).astype(np.float32))
    e = np.exp(k[1, :, 0].astype(np.float64) * D ** -0.5)
    v[0] = 1.0
    left = np.repeat(-1.0 / e[:, None], D, 1)
    for t in range(1, 5):
        v[t] = orc.round_bf16(left.astype(np.float32))
        left -= v[t]
    dev = lambda a: xh.DeviceBuffer.from_numpy(np.ascontiguousarray(a))
    bits = lambda a: dev(orc.to_bf16(a))
    dq, dk, dv, dkc, dvc = bits(q), bits(k[4:]), bits(v[4:]), bits(k), bits(v)
    dt, dc, ds, out = dev(np.zeros((1, 1), np.int32)), dev(np.asarray([4], np.int32)), dev(np.asarray([4], np.int32)), xh.DeviceBuffer(H * D * 2)
    xh.paged_attention_decode(out.ptr, dq.ptr, dk.ptr, dv.ptr, H, H, D, H * D, H * D, H * D, D ** -0.5, 1, dkc.ptr, dvc.ptr, 1, 5, dt.ptr, 1, dc.ptr, ds.ptr, 4)
    xh.synchronize()
    got = orc.from_bf16(out.to_numpy(np.uint16, (H, D))).astype(np.float64)
    p = np.stack([np.ones(H)] + [e] * 4)[:, :, None] / (1.0 + 4.0 * e)[None, :, None]
    ref, size = (p * v).sum(0), (p * np.abs(v)).sum(0)
    worst = float((np.abs(got - ref) / (np.abs(ref) * 2.0 ** -8 + size * 2.0 ** -20)).max())
    print(f"paged decode, values that cancel: {worst:.3f} of the bound", flush=True)
    assert worst <= 1.0


@pytest.mark.parametrize("qH,kvH,n", [(8, 2, 5), (8, 2, 32), (32, 8, 33), (20, 1, 700), (4, 4, 4000)])
def test_paged_decode_infinite_values(xh, orc, qH, kvH, n):
    """Infinities and NaN among the values, at the first, the last and the highest-scored tokens: every dimension of the output is what the sum of
    fp32 products gives (infinite with one sign, NaN with both or beside a NaN, finite where all values are)."""
    marks = {0: np.inf, 1: -np.inf, 2: np.nan}

    def change(v, where, b):
        for t, d in ((0, 3), (n - 1, 5), (n // 2, 6)):
            v[where[t], :, 4 * d + b % 3] = marks[b % 3]
        v[where[:], :, 70] = np.inf  # (all tokens: the highest-scored one of every head among them)
        v[where[0], :, 71], v[where[n - 1], :, 71] = np.inf, -np.inf if n > 1 else np.inf

    rng = np.random.default_rng(n)
    got, ref, size, slack = _decode64(xh, orc, rng, [n - 1] * 3, qH, kvH, change)
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isinf(got), np.isinf(ref))
    assert np.array_equal(got[np.isinf(got)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    assert (np.abs(got[fine] - ref[fine]) <= np.abs(ref[fine]) * 2.0 ** -8 + size[fine] * slack[fine]).all()


@pytest.mark.parametrize("qH,kvH,lens,block_size", [(32, 4, [33, 500, 1, 700, 65], 16), (16, 4, [31, 32, 33, 64, 96, 97], 5), (8, 8, [40] * 70, 16),
                                                    (24, 3, [600, 200, 450, 20, 7], 16), (4, 2, [3, 90, 17], 4)])
def test_paged_prefill_side_by_side(xh, orc, qH, kvH, lens, block_size):
    """Sequences that share a launch: unequal lengths about the 32-token block, more sequences than a launch takes, (sequence, KV head)
    pairs that do not divide among eight, and so little work that the 16-column form runs."""
    test_paged_prefill_matches_oracle(xh, orc, qH, kvH, lens, block_size)


@pytest.mark.parametrize("qH,kvH,lens", [(20, 5, [700, 33, 650, 500, 1, 90, 300, 64, 700]), (32, 8, [300, 700, 40, 41, 600]), (16, 8, [200] * 9),
                                         (12, 3, [400] * 3 + [10] * 20), (8, 8, [600, 300, 20, 130])])
def test_paged_prefill_bands(xh, orc, qH, kvH, lens):
    """Several groups of 8 (sequence, KV head) pairs, walked in bands by the length of the walk: a group with pairs of two sequences, lengths that are equal and
    far apart, several bands."""
    test_paged_prefill_matches_oracle(xh, orc, qH, kvH, lens, 16)


@pytest.mark.parametrize("qH,kvH,lens", [(32, 8, [1700, 1103, 33, 701]), (24, 24, [2101, 1500])])
def test_paged_prefill_that_fills_the_device(xh, orc, qH, kvH, lens):
    """Enough long walks for the form in 16 x 16 MFMAs, a short sequence beside them."""
    assert xh.paged_attention_prefill_forms(qH, kvH, lens) == [0 if n < 100 else 2 for n in lens]
    test_paged_prefill_matches_oracle(xh, orc, qH, kvH, lens, 16)


@pytest.mark.parametrize("qH,kvH,lens", [(32, 8, [200] * 8), (32, 8, [511, 150, 512, 600, 130]), (16, 4, [500, 270, 300, 20, 400]), (8, 8, [40] * 70)])
@pytest.mark.parametrize("size,key,scale", [(24.0, 1.0, 128 ** -0.5), (1.5e-4, 1e4, 128 ** -0.5), (1.0, 1e4, 1.5e-5)])
def test_paged_prefill_as_exact_as_alone(xh, orc, qH, kvH, lens, size, key, scale):
    """A sequence among others is as near to the 64-bit result as in a call of its own (2 % for another order of the sums): the same roundings of
    queries, probabilities and results, whatever else there is to do.  Large scores show a rounding of the queries: one of 2^-12 moves
    scores of 40 by 4e-3, and with them their probabilities; so do small queries, or a small scale, and keys near the end of the range."""
    D, T, rng = 128, sum(lens), np.random.default_rng(len(lens))
    q, k, v = (orc.round_bf16(rng.standard_normal((T, n, D)).astype(np.float32) * by) for n, by in ((qH, size), (kvH, key), (kvH, 1.0)))
    dq, dk, dv = (xh.DeviceBuffer.from_numpy(orc.to_bf16(a)) for a in (q, k, v))
    ds = xh.DeviceBuffer.from_numpy(np.arange(T, dtype=np.int32))
    dkc, dvc = xh.DeviceBuffer(T * kvH * D * 2), xh.DeviceBuffer(T * kvH * D * 2)
    out, one = xh.DeviceBuffer(T * qH * D * 2), xh.DeviceBuffer(T * qH * D * 2)

    def call(to, at, n):
        p = lambda buf, width: C.c_void_p(buf.ptr.value + at * width)
        xh.paged_attention_prefill(p(to, qH * D * 2), p(dq, qH * D * 2), p(dk, kvH * D * 2), p(dv, kvH * D * 2), qH, kvH, D, qH * D, kvH * D, qH * D,
                                   scale, n, dkc.ptr, dvc.ptr, T, 1, p(ds, 4))

    starts = np.concatenate([[0], np.cumsum(lens)])
    call(out, 0, lens)
    for at, n in zip(starts, lens):
        call(one, int(at), [n])
    xh.synchronize()
    together, alone = (orc.from_bf16(b.to_numpy(np.uint16, (T, qH, D))).astype(np.float64) for b in (out, one))
    for at, n in zip(starts, lens):
        off = []
        for h in range(qH):
            x = q[at:at + n, h].astype(np.float64) @ k[at:at + n, h * kvH // qH].astype(np.float64).T * scale
            x[np.triu_indices(n, 1)] = -np.inf
            p = np.exp(x - x.max(1, keepdims=True))
            ref = p / p.sum(1, keepdims=True) @ v[at:at + n, h * kvH // qH].astype(np.float64)
            off.append([np.sum((a[at:at + n, h] - ref) ** 2) for a in (together, alone)])
        a, b = np.sqrt(np.sum(off, 0))
        assert a <= 1.02 * b, f"{n} tokens: error among others / alone {a / b:.4f}"


# rows of q | k | v in one buffer; the results over the queries in place, at the buffer's start in a row length of their own, and one head on
@pytest.mark.parametrize("o_stride,shift", [(None, 0), (16, 0), (24, 1), (None, 1), (None, 16)])
@pytest.mark.parametrize("phase,B", [("decode", 3), ("decode", 70), ("prompt", 3), ("prompt", 70)])
def test_paged_results_over_their_inputs(xh, orc, phase, B, o_stride, shift):
    """Results that lie over the call's queries, keys or values, in their rows or others', are those of a call with a buffer of their own."""
    D, qH, kvH, rng = 128, 16, 4, np.random.default_rng(B)
    lens = [1] * B if phase == "decode" else [int(n) for n in rng.integers(1, 60, B)]
    T, stride, n = sum(lens), (qH + 2 * kvH) * D, 40
    o = stride if o_stride is None else o_stride * D
    rows = orc.to_bf16(_bf(orc, rng, (T + 2, stride)))
    dev = lambda a: xh.DeviceBuffer.from_numpy(a)
    kc, vc = (dev(orc.to_bf16(_bf(orc, rng, (max(B * n, T), kvH * D)))) for _ in range(2))
    slots = dev(np.arange(1, B + 1, dtype=np.int32) * n - 1 if phase == "decode" else np.arange(T, dtype=np.int32))
    table, ctx = dev(np.arange(B, dtype=np.int32)), dev(np.full(B, n - 1, np.int32))

    def call(buf, out, o):
        at = lambda heads: C.c_void_p(buf.ptr.value + heads * D * 2)
        if phase == "decode":
            xh.paged_attention_decode(out, at(0), at(qH), at(qH + kvH), qH, kvH, D, stride, stride, o, D ** -0.5, B, kc.ptr, vc.ptr, B, n, table.ptr, 1,
                                      ctx.ptr, slots.ptr, n - 1)
        else:
            xh.paged_attention_prefill(out, at(0), at(qH), at(qH + kvH), qH, kvH, D, stride, stride, o, D ** -0.5, lens, kc.ptr, vc.ptr, T, 1, slots.ptr)
        xh.synchronize()

    own, buf = xh.DeviceBuffer(T * qH * D * 2), dev(rows)
    call(buf, own.ptr, qH * D)
    want = own.to_numpy(np.uint16, (T, qH * D))
    call(buf, C.c_void_p(buf.ptr.value + shift * D * 2), o)
    flat = buf.to_numpy(np.uint16, ((T + 2) * stride,))
    got = np.stack([flat[shift * D + t * o:shift * D + t * o + qH * D] for t in range(T)])
    assert np.array_equal(got, want)


_streams = []


def _stream(xh):
    """One no test before has used: scratch is kept by a stream's handle, which a destroyed one's successor may get."""
    _streams.append(xh.Stream())
    return _streams[-1]


def _captured(xh, stream, call, out, shape):
    """Three replays of `call(stream)` captured on `stream`, each into a cleared output."""
    graph = C.c_void_p()
    xh.check(xh.lib.xfthip_graph_begin(stream.h))
    call(stream.h)
    xh.check(xh.lib.xfthip_graph_end(stream.h, C.byref(graph)))
    for _ in range(3):
        out.upload(np.zeros(shape, np.uint16))
        xh.check(xh.lib.xfthip_graph_launch(graph, stream.h))
        xh.synchronize()
        yield out.to_numpy(np.uint16, shape)
    xh.lib.xfthip_graph_destroy(graph)


def test_paged_decode_captured_behind_an_unsplit_call(xh, orc):
    """A stream's first call brings all its buffers: one that splits no context, then, captured, one that does."""
    D, qH, kvH, B, n = 128, 32, 8, 32, 300
    rng = np.random.default_rng(1)
    dev = lambda a: xh.DeviceBuffer.from_numpy(a)
    bits = lambda *shape: dev(orc.to_bf16(_bf(orc, rng, shape)))
    q, k, v, kc, vc = bits(B, qH * D), bits(B, kvH * D), bits(B, kvH * D), bits(B * n, kvH * D), bits(B * n, kvH * D)
    table, ctx, slots = dev(np.arange(B, dtype=np.int32)), dev(np.full(B, n - 1, np.int32)), dev(np.arange(1, B + 1, dtype=np.int32) * n - 1)
    out = xh.DeviceBuffer(B * qH * D * 2)

    def call(batch, stream=None):
        xh.paged_attention_decode(out.ptr, q.ptr, k.ptr, v.ptr, qH, kvH, D, qH * D, kvH * D, qH * D, D ** -0.5, batch, kc.ptr, vc.ptr, B, n, table.ptr, 1,
                                  ctx.ptr, slots.ptr, n - 1, stream=stream)

    call(4)
    xh.synchronize()
    want = out.to_numpy(np.uint16, (B, qH * D))[:4].copy()
    stream = _stream(xh)
    call(B, stream.h)
    stream.synchronize()
    for got in _captured(xh, stream, lambda st: call(4, st), out, (B, qH * D)):
        assert np.array_equal(got[:4], want)


@pytest.mark.parametrize("qH,kvH,warm,lens", [(16, 4, [100], [10] * 10), (4, 1, [150] * 2, [200])])
def test_paged_prefill_captured_with_other_lengths(xh, orc, qH, kvH, warm, lens):
    """A warm-up, then, captured, no more tokens in other lengths: in ten sequences, each with a partly filled block, and in a single one, whose
    keys are split among workgroups."""
    D, T, rng = 128, sum(warm), np.random.default_rng(3)
    bits = lambda n: xh.DeviceBuffer.from_numpy(orc.to_bf16(_bf(orc, rng, (T, n * D))))
    q, k, v, kc, vc = bits(qH), bits(kvH), bits(kvH), bits(kvH), bits(kvH)
    slots, out = xh.DeviceBuffer.from_numpy(np.arange(T, dtype=np.int32)), xh.DeviceBuffer(T * qH * D * 2)

    def call(lens, stream=None):
        xh.paged_attention_prefill(out.ptr, q.ptr, k.ptr, v.ptr, qH, kvH, D, qH * D, kvH * D, qH * D, D ** -0.5, lens, kc.ptr, vc.ptr, T, 1, slots.ptr,
                                   stream=stream)

    call(lens)
    xh.synchronize()
    n = sum(lens)
    want = out.to_numpy(np.uint16, (T, qH * D))[:n].copy()
    stream = _stream(xh)
    call(warm, stream.h)
    stream.synchronize()
    for got in _captured(xh, stream, lambda st: call(lens, st), out, (T, qH * D)):
        assert np.array_equal(got[:n], want)


def test_invoke_attention_serving_loop(orc):
    """xft::invokeAttention on host buffers: prefill of two sequences, then decode steps that append to
    the paged cache; outputs against the oracle and the caller's cache arrays kept current."""
    C.CDLL(os.path.join(ROOT, "xfastertransformer_amd", "libxft_hip.so"), mode=C.RTLD_GLOBAL)
    lib = C.CDLL(os.path.join(ROOT, "xfastertransformer_amd", "libxft_layers.so"))
    fn = getattr(lib, "_ZN3xft15invokeAttentionENS_8DataTypeEPvPKvS3_S3_PiS4_iifiPKiS3_S3_S4_S4_S4_S4_ibS4_")
    P, I = C.c_void_p, C.c_int
    fn.argtypes = [I, P, P, P, P, P, P, I, I, C.c_float, I, P, P, P, P, P, P, P, I, C.c_bool, P]
    fn.restype = None
    ptr = lambda a: a.ctypes.data_as(P)
    BF16 = 1
    qH, kvH, D, bs, block_num = 32, 8, 128, 16, 24
    rng = np.random.default_rng(77)
    lens = [37, 100]
    scale = 1.0 / np.sqrt(D)
    kc_f, vc_f = np.zeros((block_num, bs, kvH, D), np.float32), np.zeros((block_num, bs, kvH, D), np.float32)
    kc_h, vc_h = orc.to_bf16(kc_f), orc.to_bf16(vc_f)  # the caller's bf16 arrays
    blocks = [[3, 9, 17, 1], [5, 2, 11, 20, 7, 14, 8, 22]]
    slot_of = lambda b, t: blocks[b][t // bs] * bs + t % bs
    # prefill
    T = sum(lens)
    q, k, v = _bf(orc, rng, (T, qH, D)), _bf(orc, rng, (T, kvH, D)), _bf(orc, rng, (T, kvH, D))
    slots = np.asarray([slot_of(b, t) for b, L in enumerate(lens) for t in range(L)], np.int32)
    out = np.zeros((T, qH * D), np.uint16)
    qb, kb, vb = orc.to_bf16(q), orc.to_bf16(k), orc.to_bf16(v)
    qs = np.asarray([T, qH, D], np.int32)
    ks = np.asarray([T, kvH, D], np.int32)
    cs = np.asarray([block_num, bs, kvH, D], np.int32)
    tl = np.asarray(lens, np.int32)
    fn(BF16, ptr(out), ptr(qb), ptr(kb), ptr(vb), ptr(qs), ptr(ks), qH * D, kvH * D, scale, 2, ptr(tl), ptr(kc_h), ptr(vc_h), ptr(cs),
       None, None, None, 0, True, ptr(slots))
    ref = orc.paged_attention_prefill(q, k, v, lens, kc_f, vc_f, slots, scale)
    got = orc.from_bf16(out).reshape(T, qH, D)
    assert np.abs(got - ref).max() <= 2e-2 and _cos(got, ref) >= 0.9999
    assert np.array_equal(orc.from_bf16(kc_h), kc_f) and np.array_equal(orc.from_bf16(vc_h), vc_f)
    # decode steps: the second sequence crosses a block boundary at 112
    ctx = np.asarray(lens, np.int32)
    for step in range(14):
        q, k, v = _bf(orc, rng, (2, qH, D)), _bf(orc, rng, (2, kvH, D)), _bf(orc, rng, (2, kvH, D))
        nums = np.asarray([(c + 1 + bs - 1) // bs for c in ctx], np.int32)
        tab = np.zeros((2, int(nums.max())), np.int32)
        for b in range(2):
            tab[b, :nums[b]] = blocks[b][:nums[b]]
        slots = np.asarray([slot_of(b, int(ctx[b])) for b in range(2)], np.int32)
        out = np.zeros((2, qH * D), np.uint16)
        qb, kb, vb = orc.to_bf16(q), orc.to_bf16(k), orc.to_bf16(v)
        qs = np.asarray([2, qH, D], np.int32)
        ks = np.asarray([2, kvH, D], np.int32)
        fn(BF16, ptr(out), ptr(qb), ptr(kb), ptr(vb), ptr(qs), ptr(ks), qH * D, kvH * D, scale, 2, None, ptr(kc_h), ptr(vc_h), ptr(cs),
           ptr(tab), ptr(nums), ptr(ctx), 0, False, ptr(slots))
        ref = orc.paged_attention_decode(q, k, v, kc_f, vc_f, tab, ctx, slots, scale)
        got = orc.from_bf16(out).reshape(2, qH, D)
        assert np.abs(got - ref).max() <= 2e-2 and _cos(got, ref) >= 0.9999, step
        assert np.array_equal(orc.from_bf16(kc_h), kc_f) and np.array_equal(orc.from_bf16(vc_h), vc_f)
        ctx = ctx + 1
