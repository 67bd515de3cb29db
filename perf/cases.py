"""The work a user of this framework has it do, as cases that can be timed and checked.

A case is a dict of plain values.  `prepare` makes what the user's program holds before the call (packed weights, caches, models, inputs),
`run` is one pass through the public entry points of xfastertransformer_amd.capi, `exact` is the same result in 64 bits from plain torch.

Families:
  gemm       one weight-only product (xfthip_gemm, xfthip_gemm_gateup_silu): 1 row (a decoded token) to some thousands (a prompt)
  attention  attention over the contiguous cache: decode of a batch at unequal positions, prompts, later portions of prompts
  paged      attention over the block-paged BF16 cache (xft::invokeAttention): decode and prompts of unequal lengths
  moe        one sparse MLP layer of the Mixtral-8x7B shape
  generate   a uniform decoder stack: the prompt pass and greedy decoding, in lockstep or as a serving loop with sequences of its own
  plan       a stack of several kinds of layers, driven in steps of unequal parts
Widths are those of the 7B / 8x7B shapes and of the layer-plan stacks that bench.py times; stacks are cut to a few layers, since every
layer of a kind costs the same."""
import ctypes as C
import math

import numpy as np
import torch

from xfastertransformer_amd import capi as xh

HEAD, VOCAB = 128, 32000
KINDS = {"int8": xh.W_INT8, "uint4": xh.W_UINT4, "nf4": xh.W_NF4, "w8a8": xh.W_W8A8, "bf16": xh.W_BF16}
NF4 = (-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
       -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0)  # the code values of QLoRA's NormalFloat4
# width, feed-forward, query heads, key / value heads of the uniform stacks
SHAPES = {"mha": (4096, 11008, 32, 32), "gqa": (4096, 14336, 32, 8)}
PLAN = {"width": 2048, "heads": 16}  # of the layer plans; the rest stands with their records below


def listed():
    return [
        # a decoded token's output projection: the smallest call there is, where launch and round trips count
        dict(name="gemm one row", family="gemm", weights="int8", form="residual", rows=1, k=4096, n=4096, zero=False),
        # a decode batch's gate / up projection over 4-bit weights
        dict(name="gemm decode batch", family="gemm", weights="uint4", form="gateup", rows=24, k=4096, n=28672, zero=True),
        # a prompt of an odd length against the up projection of the 7B shape
        dict(name="gemm prompt", family="gemm", weights="int8", form="plain", rows=2011, k=4096, n=11008, zero=False),
        # a serving batch's decode step over long contexts, every sequence at its own position, half-size cache
        dict(name="attention decode", family="attention", phase="decode", cache="int8", batch=24, tokens=6000, past=0, q_heads=32, kv_heads=8),
        # the prompts of four sequences
        dict(name="attention prompt", family="attention", phase="prompt", cache="fp16", batch=4, tokens=2000, past=0, q_heads=32, kv_heads=8),
        # the paged cache of a serving system: a decode step of many sequences, then prompts as they arrive
        dict(name="paged decode", family="paged", phase="decode", batch=32, tokens=4100, block=16, q_heads=32, kv_heads=8),
        dict(name="paged prompt", family="paged", phase="prompt", batch=6, tokens=1500, block=16, q_heads=32, kv_heads=8),
        # a prompt's pass through one sparse MLP
        dict(name="sparse mlp", family="moe", weights="int8", tokens=256),
        # one user's chat turn, and a serving loop over prompts of unequal lengths
        dict(name="generate one", family="generate", shape="mha", weights="int8", cache="fp16", batch=1, prompt=128, new=48, layers=6, serving=False),
        dict(name="generate batch", family="generate", shape="gqa", weights="int8", cache="int8", batch=12, prompt=900, new=24, layers=3, serving=True),
        # stacks of several kinds of layers: latent attention and the delta rule; grouped attention with routed experts
        dict(name="plan latent delta", family="plan", stack="pinepel", batch=4, prompt=1500, new=16),
        dict(name="plan experts", family="plan", stack="veterax", batch=16, prompt=500, new=16),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        family = rng.choice(("gemm", "gemm", "attention", "paged", "moe", "generate", "plan"))
        if family == "gemm":
            form, kind = rng.choice(("plain", "residual", "gateup")), rng.choice(sorted(KINDS))
            k, n = rng.choice(((4096, 4096), (4096, 12288), (4096, 11008), (11008, 4096), (4096, 14336), (14336, 4096), (2048, 5632), (5632, 2048)))
            if form == "gateup":
                form, n, kind = ("gateup", 2 * n, kind) if kind != "w8a8" else ("plain", n, kind)
            c = dict(family=family, weights=kind, form=form, rows=_spread(rng, 1, 4096), k=k, n=n, zero=kind in ("uint4", "w8a8") or (kind == "int8" and rng.random() < 0.3))
        elif family == "attention":
            phase, heads = rng.choice(("decode", "prompt")), rng.choice(((32, 8), (32, 32), (16, 4)))
            batch = _spread(rng, 1, 64) if phase == "decode" else _spread(rng, 1, 8)
            tokens = _spread(rng, 100, 16000) if phase == "decode" else _spread(rng, 40, 4000)
            c = dict(family=family, phase=phase, cache=rng.choice(("fp16", "int8")), batch=batch, tokens=tokens,
                     past=_spread(rng, 30, 4000) if phase == "prompt" and rng.random() < 0.3 else 0, q_heads=heads[0], kv_heads=heads[1])
        elif family == "paged":
            phase, heads = rng.choice(("decode", "prompt")), rng.choice(((32, 8), (32, 32), (16, 4)))
            batch = _spread(rng, 1, 64) if phase == "decode" else _spread(rng, 1, 12)
            tokens = _spread(rng, 30, 9000) if phase == "decode" else _spread(rng, 20, 3000)
            c = dict(family=family, phase=phase, batch=batch, tokens=tokens, block=rng.choice((4, 16, 32, 64)), q_heads=heads[0], kv_heads=heads[1])
        elif family == "moe":
            c = dict(family=family, weights=rng.choice(("int8", "uint4")), tokens=_spread(rng, 1, 1024))
        elif family == "generate":
            c = dict(family=family, shape=rng.choice(("mha", "gqa")), weights=rng.choice(sorted(KINDS)), cache=rng.choice(("fp16", "int8")),
                     batch=_spread(rng, 1, 40), prompt=_spread(rng, 20, 2048), new=_spread(rng, 4, 64), layers=rng.choice((2, 3)), serving=rng.random() < 0.5)
        else:
            c = dict(family=family, stack=rng.choice(("pinepel", "veterax")), batch=_spread(rng, 1, 24), prompt=_spread(rng, 40, 3000), new=_spread(rng, 4, 32))
        b = dict(c)
        if _cost(b) <= most and _resident(b) <= 12e9 and c not in [{k: v for k, v in x.items() if k != "name"} for x in listed()]:
            return c


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _code_bytes(kind, k, n):
    return k * n * {"int8": 1.0, "w8a8": 1.0, "uint4": 0.5, "nf4": 0.5, "bf16": 2.0}[kind] + (0 if kind == "bf16" else 4 * n)


def _kv_bytes(cache, values):
    return values * {"fp16": 2.0, "bf16": 2.0, "int8": 1.0 + 4.0 / HEAD}[cache]


def _lengths(case):
    """Tokens of every sequence: the longest is what the case names, the others lie above half of it."""
    n, top = case["batch"], case.get("prompt", case.get("tokens"))
    return [top - (top // 2) * i // max(n, 1) for i in range(n)]


def _layer_matrices(shape):
    w, f, q, kv = SHAPES[shape]
    return [(w, (q + 2 * kv) * HEAD), (q * HEAD, w), (w, 2 * f), (f, w)]


def work(case):
    f = case["family"]
    if f == "gemm":
        m, k, n = case["rows"], case["k"], case["n"]
        out = {"plain": 2 * m * n, "residual": 8 * m * n, "gateup": m * n}[case["form"]]
        return {"bytes": _code_bytes(case["weights"], k, n) + 2 * m * k + out, "flops": 2.0 * m * k * n}
    if f == "attention":
        b, t, q, kv = case["batch"], case["tokens"], case["q_heads"], case["kv_heads"]
        if case["phase"] == "decode":
            seen = sum(_lengths(case))
            return {"bytes": _kv_bytes(case["cache"], 2 * seen * kv * HEAD) + 4 * b * q * HEAD, "flops": 4.0 * seen * q * HEAD}
        pairs = b * (t * case["past"] + t * (t + 1) / 2)
        kept = _kv_bytes(case["cache"], 2 * b * (2 * t + case["past"]) * kv * HEAD)  # written for the new tokens, read for all
        return {"bytes": kept + 2 * b * t * (2 * q + 2 * kv) * HEAD, "flops": 4.0 * pairs * q * HEAD}
    if f == "paged":
        n, q, kv = _lengths(case), case["q_heads"], case["kv_heads"]
        if case["phase"] == "decode":
            return {"bytes": 4.0 * sum(n) * kv * HEAD + 4.0 * len(n) * q * HEAD, "flops": 4.0 * sum(n) * q * HEAD}
        return {"bytes": sum(n) * HEAD * (4.0 * q + 8.0 * kv), "flops": sum(2.0 * t * (t + 1) for t in n) * q * HEAD}
    if f == "moe":
        t, experts = case["tokens"], min(8, 2 * case["tokens"])
        return {"bytes": experts * (_code_bytes(case["weights"], 4096, 28672) + _code_bytes(case["weights"], 14336, 4096)) + 8.0 * t * 4096,
                "flops": 2.0 * t * 2 * 3 * 4096 * 14336}
    if f == "generate":
        w, _, q, kv = SHAPES[case["shape"]]
        mats, n, new = _layer_matrices(case["shape"]), _lengths(case) if case["serving"] else [case["prompt"]] * case["batch"], case["new"]
        stack = case["layers"] * sum(_code_bytes(case["weights"], a, b) for a, b in mats)
        passes = (len(n) if case["serving"] else 1) + new
        seen = sum(t * new + new * (new + 1) / 2 for t in n)
        head = 2.0 * w * VOCAB
        kept = _kv_bytes(case["cache"], 2 * kv * HEAD * (2 * sum(n) + seen + len(n) * new)) * case["layers"]
        per_token = case["layers"] * 2.0 * sum(a * b for a, b in mats)
        flops = per_token * (sum(n) + len(n) * new) + (2.0 * w * VOCAB) * len(n) * (1 + new)
        flops += case["layers"] * q * HEAD * (sum(2.0 * t * (t + 1) for t in n) + 4.0 * seen)
        return {"bytes": passes * (stack + head) + kept, "flops": flops}
    n, new, w = _lengths(case), case["new"], PLAN["width"]
    tokens, seen = sum(n) + len(n) * new, sum(t * new + new * (new + 1) / 2 for t in n)
    square = sum(t * (t + 1) / 2.0 for t in n)
    weights = used = 0.0
    flops = bytes_ = 0.0
    for layer, shapes in zip(*_plan_records(case)[:2]):
        sizes = {k: float(np.prod(s)) for k, s in shapes.items() if len(s) == 2 and not k.endswith(".conv")}
        routed = sum(v for k, v in sizes.items() if k.startswith("mlp.e"))
        if layer["mixer"] == xh.MIXER_GROUPED:
            share = layer["top"] / (layer["experts"] + layer["identity"])
            weights += sum(sizes.values()) - routed
            used += routed * min(1.0, share * len(n))
            flops += 2.0 * tokens * (sum(sizes.values()) - routed + routed * share) + 4.0 * (square + seen) * layer["heads"] * 128
            bytes_ += 2.0 * 2 * layer["kv_heads"] * 128 * (2 * sum(n) + seen)
            weights += routed / (1 + new)  # the prompts' step uses all of them
        else:
            weights += sum(sizes.values())
            flops += 2.0 * tokens * sum(sizes.values())
            if layer["mixer"] == xh.MIXER_LATENT:
                near = layer["window"]
                a = sum(min(t, near) * (t - min(t, near) / 2.0) if near else t * (t + 1) / 2.0 for t in n)
                s = sum(min(t, near) * new for t in n) if near else seen
                flops += 2.0 * a * layer["heads"] * 320 + 2.0 * s * layer["heads"] * (2 * 512 + 64)
                bytes_ += 2.0 * 576 * (2 * sum(n) + s)
            else:
                flops += 8.0 * tokens * layer["heads"] * 128 * 128
                bytes_ += 8.0 * layer["heads"] * 128 * 128 * len(n) * (1 + new)
    flops += 2.0 * w * VOCAB * len(n) * (1 + new)
    return {"bytes": (1 + new) * 2.0 * (weights + w * VOCAB) + new * 2.0 * used + bytes_, "flops": flops}


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 1e15


def _resident(case):
    if case["family"] == "attention":
        return case["batch"] * (case["tokens"] + case["past"]) * (case["q_heads"] + 2 * case["kv_heads"]) * HEAD * 4.0
    if case["family"] == "generate":
        return case["batch"] * (case["prompt"] + case["new"]) * 4096 * 64.0 + case["layers"] * 5e8
    return 0.0


def tolerance(case):
    """bf16 (8 bits) operands, activations and results: one rounding is 2^-9 of a value at most and 1.7e-3 in the mean square.  Measured against
    exact(): single products, attention and the sparse MLP 1.6e-3 to 2.8e-3 (int8 caches and w8a8 rows 0.7e-2 to 1e-2, single values of such
    outputs up to 0.28), stacks 0.6e-2 to 1.4e-2 (w8a8: 5e-2;
    routed experts, whose residual is mostly the embedding: 0.5e-3 to 0.8e-3).  Products
    that leave in 32 bits: int8 and bf16 codes 0.7e-7 to 3e-7, nf4 (code values in two parts) 1.4e-6, uint4 (zero points against the rows' sums) 2e-5."""
    if case.get("stack") == "veterax":
        return {"rel": 0.005, "max": 0.1}
    if case["family"] in ("generate", "plan"):
        return {"rel": 0.03, "max": 0.3, "differ": 0.0}
    if case["family"] == "moe":
        return {"rel": 0.01, "max": 0.1}
    if case.get("weights") == "w8a8" or case.get("cache") == "int8":
        return {"rel": 0.03, "max": 0.9}
    if case.get("form") == "residual":
        return {"uint4": {"rel": 8e-5, "max": 2e-3}, "nf4": {"rel": 6e-6, "max": 1e-4}}.get(case["weights"], {"rel": 2e-6, "max": 2e-5})
    return {"rel": 0.007, "max": 0.1}


# ------------------------------------------------------------------------------------------------ inputs
def _gen(seed, salt=0):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + salt)


def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _bits(t):
    """Host bf16 patterns of a tensor."""
    return t.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16)


class _Codes:
    """Codes as N(0, 0.02^2) weights quantise to, cut out of one pool at different places: weight i is the same [k, n] on the host and here."""

    def __init__(self, kind, largest, seed):
        self.kind, gen = kind, _gen(seed, 77)
        n = int(largest * (0.5 if kind in ("uint4", "nf4") else 1.0)) + (8 << 20)
        if kind in ("uint4", "nf4"):
            middles = torch.tensor([(a + b) / 2 for a, b in zip(NF4, NF4[1:])], device="cuda")
            if kind == "nf4":  # the nearest code value, so that what is drawn about zero stays so
                pair = lambda: torch.bucketize(_normal(gen, n) / 3.5, middles).to(torch.uint8)
            else:
                pair = lambda: (_normal(gen, n) * (15.0 / 8.4) + 7.5).round_().clamp_(0, 15).to(torch.uint8)
            self.pool = pair() | (pair() << 4)
        elif kind == "bf16":
            self.pool = (_normal(gen, n) * 0.02).to(torch.bfloat16)
        else:
            self.pool = (_normal(gen, n) * (127.0 / 4.2)).round_().clamp_(-127, 127).to(torch.int8)
        self.host = self.pool.view(torch.int16).cpu().numpy().view(np.uint16) if kind == "bf16" else self.pool.cpu().numpy()
        self.seed = seed

    def _at(self, i, count):
        return (i * 1299709 * 16) % (len(self.pool) - count + 1)

    def _columns(self, i, n, zero):
        rng = np.random.default_rng((self.seed, 5, i))
        step = {"int8": 0.02 * 4.2 / 127, "w8a8": 0.02 * 4.2 / 127, "uint4": 0.02 * 8.4 / 15, "nf4": 0.02 * 3.5, "bf16": 1.0}[self.kind]
        scale = (step * rng.uniform(0.75, 1.25, n)).astype(np.float32)
        if self.kind == "uint4":
            return scale, (-7.5 * scale + 0.002 * rng.standard_normal(n)).astype(np.float32)
        return scale, (0.001 * rng.standard_normal(n)).astype(np.float32) if zero and self.kind != "nf4" else None

    def weight(self, i, k, n, zero=False, gateup=False):
        flags = xh.WF_GATEUP if gateup else xh.WF_NONE
        count = k * n // (2 if self.kind in ("uint4", "nf4") else 1)
        at = self._at(i, count)
        q = self.host[at:at + count].reshape(k, -1)
        if self.kind == "bf16":
            return xh.Weight(xh.W_BF16, k, n, q, flags=flags)
        scale, z = self._columns(i, n, zero)
        return xh.Weight(KINDS[self.kind], k, n, q, scale, z, flags=flags)

    def dense(self, i, k, n, zero=False):
        count = k * n // (2 if self.kind in ("uint4", "nf4") else 1)
        at = self._at(i, count)
        q = self.pool[at:at + count].reshape(k, -1)
        if self.kind == "bf16":
            return q.double()
        if self.kind in ("uint4", "nf4"):
            q = torch.stack((q & 15, q >> 4), -1).reshape(k, n)
        scale, z = self._columns(i, n, zero)
        scale = torch.from_numpy(scale).cuda().double()
        if self.kind == "nf4":
            return torch.tensor(NF4, dtype=torch.float32, device="cuda").double()[q.long()] * scale
        return q.double() * scale + (0.0 if z is None else torch.from_numpy(z).cuda().double())


def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, past, scale, window=0, sink=None):
    """q [s, heads, d], k and v [t, kv heads, d] in 64 bits; query i sees keys up to past + i."""
    s, t, share = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    i, j = torch.arange(s, device="cuda")[:, None] + past, torch.arange(t, device="cuda")[None, :]
    hidden = (j > i) | (i - j >= (window or t + s))
    out = torch.empty(s, q.shape[1], v.shape[2], dtype=torch.float64, device="cuda")
    for h in range(q.shape[1]):
        x = (q[:, h] @ k[:, h // share].T * scale).masked_fill_(hidden, -math.inf)
        if sink is not None:
            x = torch.cat((x, sink[h].expand(s, 1)), 1)
        out[:, h] = torch.softmax(x, 1)[:, :t] @ v[:, h // share]
    return out


def _turn(x, start, base, dims, interleaved, freq=None, mul=1.0):
    """x [t, heads, n]: its first `dims` entries turned by their position."""
    half = dims // 2
    f = float(base) ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / dims) if freq is None else freq
    a = (start + torch.arange(x.shape[0], dtype=torch.float64, device="cuda"))[:, None] * f
    c, s = torch.cos(a)[:, None] * mul, torch.sin(a)[:, None] * mul
    y = x.clone()
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if interleaved else (x[..., :half], x[..., half:dims])
    if interleaved:
        y[..., 0:dims:2], y[..., 1:dims:2] = u * c - v * s, v * c + u * s
    else:
        y[..., :half], y[..., half:dims] = u * c - v * s, v * c + u * s
    return y


def prepare(case, seed):
    xh.init()
    return {"case": case, **globals()["_prepare_" + case["family"]](case, seed)}


def run(state):
    return globals()["_run_" + state["case"]["family"]](state["case"], state)


def exact(case, seed):
    return globals()["_exact_" + case["family"]](case, seed)


# ------------------------------------------------------------------------------------------------ one product
def _gemm_inputs(case, seed):
    gen = _gen(seed)
    return _normal(gen, case["rows"], case["k"]).to(torch.bfloat16), _normal(gen, case["rows"], case["n"]) if case["form"] == "residual" else None


def _prepare_gemm(case, seed):
    m, n = case["rows"], case["n"]
    a, res = _gemm_inputs(case, seed)
    out = torch.empty(m, n // 2 if case["form"] == "gateup" else n, device="cuda", dtype=torch.float32 if res is not None else torch.bfloat16)
    w = _Codes(case["weights"], case["k"] * n, seed).weight(0, case["k"], n, case["zero"], case["form"] == "gateup")
    return {"a": a, "res": res, "out": out, "w": w}


def _run_gemm(case, s):
    m, k, n, a, out = case["rows"], case["k"], case["n"], s["a"], s["out"]
    if case["form"] == "gateup":
        xh.gemm_gateup_silu(s["w"], _ptr(a), m, k, _ptr(out), n // 2, xh.BF16)
    elif case["form"] == "residual":
        xh.gemm(s["w"], _ptr(a), m, k, _ptr(out), n, xh.F32, epi=xh.EPI_RESIDENTIAL, res=_ptr(s["res"]), ldres=n, res_dtype=xh.F32)
    else:
        xh.gemm(s["w"], _ptr(a), m, k, _ptr(out), n, xh.BF16)
    return out


def _exact_gemm(case, seed):
    a, res = _gemm_inputs(case, seed)
    y = a.double() @ _Codes(case["weights"], case["k"] * case["n"], seed).dense(0, case["k"], case["n"], case["zero"])
    if case["form"] == "gateup":
        half = case["n"] // 2
        return _silu(y[:, :half]) * y[:, half:]
    return y if res is None else y + res.double()


# ------------------------------------------------------------------------------------------------ attention over the contiguous cache
def _fill(case, cache, seed, total):
    """Keys and values of `total` tokens a sequence, in portions as a prompt brings them; the portions' rows are made again by exact()."""
    q, kv, b = case["q_heads"], case["kv_heads"], case["batch"]
    for at in range(0, total, 512):
        s = min(512, total - at)
        rows = _portion(case, seed, at, s)
        full = torch.zeros(b * s, (q + 2 * kv) * HEAD, dtype=torch.bfloat16, device="cuda")
        full[:, q * HEAD:] = rows
        xh.rope_kvstore(cache, _ptr(full), xh.BF16, full.shape[1], b, s, q, None, at)
        torch.cuda.synchronize()


def _portion(case, seed, at, s):
    return _normal(_gen(seed, 1000 + at), case["batch"] * s, 2 * case["kv_heads"] * HEAD).to(torch.bfloat16)


def _kept(case, seed, total):
    """[batch, total, 2, kv heads, HEAD] of what _fill stored."""
    parts = [_portion(case, seed, at, min(512, total - at)).reshape(case["batch"], -1, 2, case["kv_heads"], HEAD) for at in range(0, total, 512)]
    return torch.cat(parts, 1)


def _prepare_attention(case, seed):
    b, t, q, kv = case["batch"], case["tokens"], case["q_heads"], case["kv_heads"]
    decode, past = case["phase"] == "decode", case["past"]
    cache = xh.KVCache(xh.INT8 if case["cache"] == "int8" else xh.FP16, b, kv, t + past, HEAD)
    s = {"cache": cache}
    if decode:
        _fill(case, cache, seed, t)
        s["q"] = _normal(_gen(seed, 3), b, q * HEAD).to(torch.bfloat16)
        s["positions"] = torch.tensor([n - 1 for n in _lengths(case)], dtype=torch.int32, device="cuda")
        s["out"] = torch.empty(b, q * HEAD, dtype=torch.bfloat16, device="cuda")
    else:
        _fill(case, cache, seed, past)
        s["qkv"] = _normal(_gen(seed, 3), b * t, (q + 2 * kv) * HEAD).to(torch.bfloat16)
        s["out"] = torch.empty(b * t, q * HEAD, dtype=torch.bfloat16, device="cuda")
    return s


def _run_attention(case, s):
    b, t, q, kv = case["batch"], case["tokens"], case["q_heads"], case["kv_heads"]
    if case["phase"] == "decode":
        xh.attention(s["cache"], _ptr(s["q"]), q * HEAD, _ptr(s["out"]), q * HEAD, xh.BF16, b, 1, q, HEAD ** -0.5, t - 1, _ptr(s["positions"]))
    else:
        stride = (q + 2 * kv) * HEAD
        xh.rope_kvstore(s["cache"], _ptr(s["qkv"]), xh.BF16, stride, b, t, q, None, case["past"])
        xh.attention(s["cache"], _ptr(s["qkv"]), stride, _ptr(s["out"]), q * HEAD, xh.BF16, b, t, q, HEAD ** -0.5, case["past"])
    return s["out"]


def _exact_attention(case, seed):
    b, t, q, kv, past = case["batch"], case["tokens"], case["q_heads"], case["kv_heads"], case["past"]
    if case["phase"] == "decode":
        rows, x = _kept(case, seed, t), _normal(_gen(seed, 3), b, q * HEAD).to(torch.bfloat16).double().reshape(b, 1, q, HEAD)
        got = [_attend(x[i], rows[i, :n, 0].double(), rows[i, :n, 1].double(), n - 1, HEAD ** -0.5) for i, n in enumerate(_lengths(case))]
        return torch.cat(got).reshape(b, q * HEAD)
    x = _normal(_gen(seed, 3), b * t, (q + 2 * kv) * HEAD).to(torch.bfloat16).reshape(b, t, q + 2 * kv, HEAD)
    old = _kept(case, seed, past) if past else x.new_zeros(b, 0, 2, kv, HEAD)
    out = []
    for i in range(b):
        k, v = torch.cat((old[i, :, 0], x[i, :, q:q + kv])).double(), torch.cat((old[i, :, 1], x[i, :, q + kv:])).double()
        out.append(_attend(x[i, :, :q].double(), k, v, past, HEAD ** -0.5).reshape(t, q * HEAD))
    return torch.cat(out)


# ------------------------------------------------------------------------------------------------ attention over the paged cache
def _paged_inputs(case, seed):
    """Lengths (the new token included in decoding), block tables, caches and the new rows."""
    n, kv, q, block = _lengths(case), case["kv_heads"], case["q_heads"], case["block"]
    need = [-(-t // block) for t in n]
    blocks = sum(need) + 8
    order = np.random.default_rng((seed, 11)).permutation(blocks).astype(np.int32)
    table, at = np.zeros((len(n), max(need)), np.int32), 0
    for b, c in enumerate(need):
        table[b, :c] = order[at:at + c]
        at += c
    gen, decode = _gen(seed, 3), case["phase"] == "decode"
    rows = len(n) if decode else sum(n)
    make = lambda: _normal(gen, blocks, block, kv, HEAD).to(torch.bfloat16)
    s = {"k_cache": make(), "v_cache": make(), "q": _normal(gen, rows, q * HEAD).to(torch.bfloat16),
         "k": _normal(gen, rows, kv * HEAD).to(torch.bfloat16), "v": _normal(gen, rows, kv * HEAD).to(torch.bfloat16)}
    slot = lambda b, t: table[b, t // block] * block + t % block
    slots = [slot(b, t - 1) for b, t in enumerate(n)] if decode else np.concatenate([slot(b, np.arange(t)) for b, t in enumerate(n)])
    return n, table, np.asarray(slots, np.int32), blocks, s


def _prepare_paged(case, seed):
    n, table, slots, blocks, s = _paged_inputs(case, seed)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.int32)).cuda()
    s.update(lengths=n, table=up(table), slots=up(slots), contexts=up([t - 1 for t in n]), blocks=blocks, out=torch.empty_like(s["q"]))
    return s


def _run_paged(case, s):
    q, kv, block, n = case["q_heads"], case["kv_heads"], case["block"], s["lengths"]
    if case["phase"] == "decode":
        xh.paged_attention_decode(_ptr(s["out"]), _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), q, kv, HEAD, q * HEAD, kv * HEAD, q * HEAD, HEAD ** -0.5, len(n),
                                  _ptr(s["k_cache"]), _ptr(s["v_cache"]), s["blocks"], block, _ptr(s["table"]), s["table"].shape[1], _ptr(s["contexts"]),
                                  _ptr(s["slots"]), max(n) - 1)
    else:
        xh.paged_attention_prefill(_ptr(s["out"]), _ptr(s["q"]), _ptr(s["k"]), _ptr(s["v"]), q, kv, HEAD, q * HEAD, kv * HEAD, q * HEAD, HEAD ** -0.5, n,
                                   _ptr(s["k_cache"]), _ptr(s["v_cache"]), s["blocks"], block, _ptr(s["slots"]))
    return {"out": s["out"], "k_cache": s["k_cache"], "v_cache": s["v_cache"]}


def _exact_paged(case, seed):
    n, table, slots, _, s = _paged_inputs(case, seed)
    q, kv, block = case["q_heads"], case["kv_heads"], case["block"]
    for c, new in (("k_cache", "k"), ("v_cache", "v")):
        s[c].view(-1, kv * HEAD)[torch.from_numpy(slots).cuda().long()] = s[new]
    out, at = [], 0
    for b, t in enumerate(n):
        where = torch.from_numpy(table[b, :-(-t // block)]).cuda().long()
        k, v = (s[c][where].reshape(-1, kv, HEAD)[:t].double() for c in ("k_cache", "v_cache"))
        rows = 1 if case["phase"] == "decode" else t
        out.append(_attend(s["q"][at:at + rows].double().reshape(rows, q, HEAD), k, v, t - rows, HEAD ** -0.5).reshape(rows, q * HEAD))
        at += rows
    return {"out": torch.cat(out), "k_cache": s["k_cache"].double(), "v_cache": s["v_cache"].double()}


# ------------------------------------------------------------------------------------------------ sparse MLP
def _moe_inputs(case, seed):
    """Tokens that lean towards two experts each, as those of a trained router do: no near ties."""
    gen, t = _gen(seed), case["tokens"]
    router = _normal(gen, 4096, 8) * 0.05
    pick = torch.rand(t, 8, generator=gen, device="cuda").argsort(1)[:, :2]
    lean = router.T / router.T.norm(dim=1, keepdim=True)
    x = _normal(gen, t, 4096) + 30.0 * lean[pick[:, 0]] + 18.0 * lean[pick[:, 1]]
    return router, x, (1.0 + 0.1 * _normal(gen, 4096))


def _prepare_moe(case, seed):
    router, x, norm = _moe_inputs(case, seed)
    codes = _Codes(case["weights"], 4096 * 28672, seed)
    moe = xh.MoE(4096, 14336, 8, max(case["tokens"], 32), router.cpu().numpy(), norm.cpu().numpy())
    for e in range(8):
        moe.set_expert(e, codes.weight(2 * e, 4096, 28672, gateup=True), codes.weight(2 * e + 1, 14336, 4096))
    return {"moe": moe, "x": x, "out": torch.empty_like(x)}


def _run_moe(case, s):
    s["moe"].forward(_ptr(s["x"]), _ptr(s["out"]), case["tokens"], want_routing=False)
    return s["out"]


def _exact_moe(case, seed):
    router, x, norm = (t.double() for t in _moe_inputs(case, seed))
    codes, xn, out = _Codes(case["weights"], 4096 * 28672, seed), _rms(x) * norm, x.clone()
    top, which = (xn @ router).topk(2, 1)
    share = torch.softmax(top, 1)
    for e in range(8):
        t, slot = (which == e).nonzero(as_tuple=True)
        if len(t):
            y = xn[t] @ codes.dense(2 * e, 4096, 28672)
            out[t] += share[t, slot][:, None] * ((_silu(y[:, :14336]) * y[:, 14336:]) @ codes.dense(2 * e + 1, 14336, 4096))
    return out


# ------------------------------------------------------------------------------------------------ uniform stacks
def _stack_inputs(case, seed):
    """Embedding, head and prompts.  The head answers a token with its successor in a permutation, by a margin that layers of
    random weights do not bridge: what is generated is the same whatever the order of sums."""
    w, gen = SHAPES[case["shape"]][0], _gen(seed, 9)
    embed = _normal(gen, VOCAB, w).half()
    after = torch.randperm(VOCAB, generator=gen, device="cuda")
    head = torch.empty(VOCAB, w, dtype=torch.bfloat16, device="cuda")
    head[after] = (embed.float() * 0.02).to(torch.bfloat16)
    n = _lengths(case) if case["serving"] else [case["prompt"]] * case["batch"]
    ids = [torch.randint(0, VOCAB, (t,), generator=gen, device="cuda") for t in n]
    return embed, after, head, ids


def _stack_weights(case, seed):
    return _Codes(case["weights"], max(a * b for a, b in _layer_matrices(case["shape"])), seed)


def _prepare_generate(case, seed):
    w, f, q, kv = SHAPES[case["shape"]]
    embed, _, head, ids = _stack_inputs(case, seed)
    codes, ones = _stack_weights(case, seed), np.ones(w, np.float32)
    top = max(len(i) for i in ids)
    model = xh.Model(case["layers"], w, f, q, kv, HEAD, vocab=VOCAB, max_batch=case["batch"], max_seq=top + case["new"] + 1,
                     max_tokens=top if case["serving"] else top * case["batch"], kv_dtype=xh.INT8 if case["cache"] == "int8" else xh.FP16)
    zero = case["weights"] in ("uint4", "w8a8")
    for l in range(case["layers"]):
        model.set_layer(l, *[codes.weight(4 * l + i, a, b, zero, i == 2 and case["weights"] != "w8a8") for i, (a, b) in enumerate(_layer_matrices(case["shape"]))], ones, ones)
    model.set_head(embed.view(torch.int16).cpu().numpy().view(np.uint16), ones, xh.Weight(xh.W_BF16, w, VOCAB, _bits(head.T.contiguous())))
    return {"model": model, "ids": [i.cpu().numpy().astype(np.int32) for i in ids]}


def _run_generate(case, s):
    model, ids, b, new = s["model"], s["ids"], case["batch"], case["new"]
    if not case["serving"]:
        _, first = model.prefill(np.stack(ids), want_logits=True)
        tokens = model.decode(new, b)
        return {"first": first, "tokens": tokens, "last": model.logits(b)}
    rows = list(range(b))
    first = np.stack([model.seq_prefill(r, ids[r], want_logits=True) for r in rows])
    tokens = np.stack([model.seq_decode(rows) for _ in range(new)])
    last = np.stack([model.seq_logits(r) for r in rows])
    for r in rows:
        model.seq_release(r)
    return {"first": first, "tokens": tokens, "last": last}


def _exact_generate(case, seed):
    w, f, q, kv = SHAPES[case["shape"]]
    embed, after, head, ids = _stack_inputs(case, seed)
    codes, new, zero = _stack_weights(case, seed), case["new"], case["weights"] in ("uint4", "w8a8")
    whole = []
    for i in ids:  # the last step reads the token in front of the last one generated
        chain = [after[i[-1]]]
        for _ in range(new - 1):
            chain.append(after[chain[-1]])
        whole.append(torch.cat((i, torch.stack(chain))))
    x, at = embed[torch.cat(whole)].double(), np.cumsum([0] + [len(i) for i in whole])
    for l in range(case["layers"]):
        d = lambda i: codes.dense(4 * l + i, *_layer_matrices(case["shape"])[i], zero)
        y, o = (_rms(x) @ d(0)).reshape(len(x), q + 2 * kv, HEAD), []
        for b in range(len(ids)):
            z = y[at[b]:at[b + 1]]
            o.append(_attend(_turn(z[:, :q], 0, 10000, HEAD, False), _turn(z[:, q:q + kv], 0, 10000, HEAD, False), z[:, q + kv:], 0, HEAD ** -0.5))
        x = x + torch.cat(o).reshape(len(x), q * HEAD) @ d(1)
        y = _rms(x) @ d(2)
        x = x + (_silu(y[:, :f]) * y[:, f:]) @ d(3)
    logits = lambda rows: _rms(x[rows]) @ head.double().T
    first = logits([int(at[b]) + len(i) - 1 for b, i in enumerate(ids)])
    return {"first": first, "tokens": None, "last": logits([int(e) - 1 for e in at[1:]])}


# ------------------------------------------------------------------------------------------------ layer plans
def _plan_records(case):
    """(records, tensor shapes of each, arguments of the plan) of the stacks that bench.py times at width 2048, each kind of layer once
    (pinepel: windowed latent attention, latent attention with a sink, the delta rule) or two layers (veterax)."""
    w, h = PLAN["width"], PLAN["heads"]
    if case["stack"] == "pinepel":
        ff = dict(inter=5632, glu_limit=7.0, glu_alpha=1.702)
        latent = dict(mixer=xh.MIXER_LATENT, heads=h, dim=128, vdim=128, rot_dim=64, kv_rank=512, q_rank=768, scale=192 ** -0.5, rot_base=1e6, window=0, **ff)
        records = [dict(latent, rot_interleaved=1, window=1024), dict(latent, has_sink=1),
                   dict(mixer=xh.MIXER_DELTA, heads=h, kv_heads=h, dim=128, vdim=128, taps=4, decay_rank=128, gate_rank=128, **ff)]
        both = {n: (w,) for n in ("norm1", "norm1b", "ls1", "norm2", "norm2b", "ls2")}
        both.update({"mlp.gate": (5632, w), "mlp.up": (5632, w), "mlp.down": (w, 5632), "mix.o": (w, h * 128)})
        lat = {"mix.dq": (768, w), "mix.dq.norm": (768,), "mix.uq": (h * 192, 768), "mix.dkv": (576, w), "mix.dkv.norm": (512,), "mix.uk": (h * 128, 512),
               "mix.uv": (h * 128, 512)}
        d = h * 128
        delta = {"mix.b": (h, w), "mix.A_log": (h,), "mix.norm": (128,), "mix.a1": (128, w), "mix.a2": (d, 128), "mix.dt_bias": (d,), "mix.g1": (128, w),
                 "mix.g2": (d, 128)}
        for n in "qkv":
            delta["mix." + n], delta["mix." + n + ".conv"] = (d, w), (d, 4)
        return records, [dict(both, **lat), dict(both, **lat, **{"mix.sink": (h,)}), dict(both, **delta)], {}
    kv, side = 4, 256
    layer = dict(mixer=xh.MIXER_GROUPED, heads=h, kv_heads=kv, dim=128, vdim=128, rot_dim=128, rot_interleaved=1, rot_base=1e6, rot_factor=4.0, rot_original=8192,
                 rot_fast=32.0, rot_slow=1.0, scale=128 ** -0.5, has_sink=1, qk_norm=1, v_mix=1, inter=2816, glu_limit=7.0, glu_alpha=1.702, experts=8, identity=2,
                 top=2, expert_inter=2816, expert_limit=7.0)
    t = {"mix.q": (h * 128, w), "mix.k": (kv * 128, w), "mix.v": (kv * 128, w), "mix.q.norm": (128,), "mix.k.norm": (128,), "mix.sink": (h,), "mix.vmix": (1,),
         "mix.o": (w, h * 128), "mlp.router": (10, w), "mlp.correction": (10,), "side.gate": (side, w), "side.proj": (w, side), "side.norm": (w,)}
    for n in ("norm1", "norm2"):
        t[n], t[n + ".b"], t[n + ".alpha"] = (w,), (w,), (1,)
    for p in ["e%d." % e for e in range(8)] + ["shared."]:
        t["mlp." + p + "gate"], t["mlp." + p + "up"], t["mlp." + p + "down"] = (2816, w), (2816, w), (w, 2816)
    return [layer] * 2, [t] * 2, dict(block=xh.BLOCK_PARALLEL, norm=xh.NORM_DYNAMIC_TANH, tied_head=1, side_dim=side)


def _plan_tensors(case, seed):
    """Every tensor by (layer, name), bf16, here: matrices keep the size of what they multiply, norms and the rest as trained ones look."""
    gen = _gen(seed, 21)
    about_one = case["stack"] == "pinepel"  # norms whose stored weights are distances from one

    def value(name, shape):
        leaf = name.split(".")[-1]
        if leaf == "alpha":
            return torch.full(shape, 0.5, device="cuda")
        if name in ("mix.dq.norm", "mix.dkv.norm", "mix.norm", "mix.q.norm", "mix.k.norm", "side.norm") or leaf in ("ls1", "ls2"):
            return 1.0 + 0.1 * _normal(gen, *shape)
        if leaf.startswith("norm"):
            return (0.0 if about_one else 1.0) + 0.1 * _normal(gen, *shape)
        if name == "mlp.router":
            return 0.012 * signs + 0.002 * _normal(gen, *shape)
        if leaf in ("b", "correction") and len(shape) == 1:
            return 0.02 * _normal(gen, *shape)
        if name in ("mix.sink", "mix.A_log", "mix.vmix"):
            return 0.5 * torch.rand(*shape, generator=gen, device="cuda")
        if name == "mix.dt_bias":
            return -3.0 + _normal(gen, *shape)
        if leaf == "conv":
            return 0.5 * _normal(gen, *shape)
        return shape[-1] ** -0.5 * _normal(gen, *shape)

    w, (records, shapes, args) = PLAN["width"], _plan_records(case)
    embed = _normal(gen, VOCAB, w)
    if not about_one:  # trained routers are sure of their choice: every token leans towards two of their outputs
        signs = _normal(gen, 10, w).sign()
        pick = torch.rand(VOCAB, 10, generator=gen, device="cuda").argsort(1)
        embed += 0.8 * signs[pick[:, 0]] + 0.6 * signs[pick[:, 1]]
    t = {(-1, "embed"): embed, (-1, "final.norm"): value("final.norm", (w,))}
    if args.get("tied_head"):
        t[-1, "final.norm.alpha"], t[-1, "final.norm.b"] = value("alpha", (1,)), value("b", (w,))
        t[-1, "side.embed"] = _normal(gen, VOCAB, args["side_dim"] * len(records))
    else:
        t[-1, "head"] = value("head", (VOCAB, w))
    for l, tensors in enumerate(shapes):
        for n, s in tensors.items():
            t[l, n] = value(n, s)
    return {k: v.to(torch.bfloat16) for k, v in t.items()}


def _plan_ids(case, seed):
    gen = _gen(seed, 22)
    return [torch.randint(0, VOCAB, (t + case["new"],), generator=gen, device="cuda") for t in _lengths(case)]


def _prepare_plan(case, seed):
    records, _, args = _plan_records(case)
    plan = xh.Plan(PLAN["width"], VOCAB, records, **args)
    for (l, n), v in _plan_tensors(case, seed).items():
        plan.set(l, n, _bits(v))
    plan.finish()
    n = _lengths(case)
    top = max(n) + case["new"]
    model = xh.PlanModel(plan, xh.BF16, len(n), top, max(sum(n), 64), sum(-(-(t + case["new"]) // 64) * 64 for t in n))
    return {"model": model, "lengths": n, "ids": [i.cpu().numpy().astype(np.int32) for i in _plan_ids(case, seed)]}


def _run_plan(case, s):
    """All prompts in one step, then one token a sequence and step, the caller choosing the tokens from the logits it is handed."""
    model, ids, n = s["model"], s["ids"], s["lengths"]
    logits = [model.step([(b, i[:t], [t - 1]) for b, (i, t) in enumerate(zip(ids, n))])]
    for k in range(case["new"]):
        logits.append(model.step([(b, i[t + k:t + k + 1], [0]) for b, (i, t) in enumerate(zip(ids, n))]))
    for b in range(len(n)):
        model.seq_release(b)
    return logits


def _glu(x, gate, up, down):
    g, u = (x @ gate.T).clamp(max=7.0), (x @ up.T).clamp(-7.0, 7.0)
    return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ down.T


def _latent(x, w, m):
    t, h = len(x), m["heads"]
    q = (_rms(x @ w("mix.dq").T) * w("mix.dq.norm")) @ w("mix.uq").T
    q, kv = q.reshape(t, h, 192), x @ w("mix.dkv").T
    c, inter = _rms(kv[:, :512]) * w("mix.dkv.norm"), bool(m.get("rot_interleaved"))
    kr = _turn(kv[:, None, 512:], 0, 1e6, 64, inter).expand(t, h, 64)
    k = torch.cat(((c @ w("mix.uk").T).reshape(t, h, 128), kr), 2)
    q = torch.cat((q[..., :128], _turn(q[..., 128:], 0, 1e6, 64, inter)), 2)
    sink = w("mix.sink") if m.get("has_sink") else None
    return _attend(q, k, (c @ w("mix.uv").T).reshape(t, h, 128), 0, m["scale"], m["window"], sink).reshape(t, h * 128) @ w("mix.o").T


def _delta(x, w, m):
    t, h = len(x), m["heads"]

    def part(n):
        y, taps = x @ w("mix." + n).T, w("mix." + n + ".conv")
        y = torch.cat((y.new_zeros(3, y.shape[1]), y))
        return _silu(sum(y[j:j + t] * taps[:, j] for j in range(4))).reshape(t, h, 128)

    unit = lambda y: y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6)
    q, k, v = unit(part("q")) * 128 ** -0.5, unit(part("k")), part("v")
    beta = torch.sigmoid(x @ w("mix.b").T)
    step = torch.nn.functional.softplus((x @ w("mix.a1").T) @ w("mix.a2").T + w("mix.dt_bias")).reshape(t, h, 128)
    g = torch.exp(-torch.exp(w("mix.A_log"))[:, None] * step)
    state, out = x.new_zeros(h, 128, 128), torch.empty_like(v)
    for i in range(t):
        state = state * g[i][:, :, None]
        u = beta[i][:, None] * (v[i] - torch.matmul(k[i][:, None], state)[:, 0])
        state = state + k[i][:, :, None] * u[:, None, :]
        out[i] = torch.matmul(q[i][:, None], state)[:, 0]
    gate = torch.sigmoid((x @ w("mix.g1").T) @ w("mix.g2").T).reshape(t, h, 128)
    return (_rms(out) * w("mix.norm") * gate).reshape(t, h * 128) @ w("mix.o").T


def _grouped(x, w, m, first):
    t, h, kv = len(x), m["heads"], m["kv_heads"]
    i = torch.arange(64, dtype=torch.float64, device="cuda")
    f = float(m["rot_base"]) ** (-2.0 * i / 128)
    turns = lambda n: 128 * math.log(m["rot_original"] / (2.0 * math.pi * n)) / (2.0 * math.log(m["rot_base"]))
    lo, hi = max(math.floor(turns(m["rot_fast"])), 0), min(math.ceil(turns(m["rot_slow"])), 127)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    f, mul = f / m["rot_factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(m["rot_factor"]) + 1.0
    q = _turn(_rms((x @ w("mix.q").T).reshape(t, h, 128)) * w("mix.q.norm"), 0, 0, 128, True, f, mul)
    k = _turn(_rms((x @ w("mix.k").T).reshape(t, kv, 128)) * w("mix.k.norm"), 0, 0, 128, True, f, mul)
    own = (x @ w("mix.v").T).reshape(t, kv, 128)
    v = own if first is None else own + w("mix.vmix") * (first - own)
    return _attend(q, k, v, 0, m["scale"], 0, w("mix.sink")).reshape(t, h * 128) @ w("mix.o").T, own


def _routed(x, w, m):
    s = torch.softmax(x @ w("mlp.router").T, 1)
    which = (s + w("mlp.correction")).topk(m["top"], 1)[1]
    share = torch.zeros_like(s).scatter_(1, which, s.gather(1, which))
    p = lambda e: [w("mlp." + e + "." + n) for n in ("gate", "up", "down")]
    y = share[:, m["experts"]:].sum(1, keepdim=True) * x + _glu(x, *p("shared"))
    for e in range(m["experts"]):
        t = share[:, e].nonzero()[:, 0]
        if len(t):
            y[t] += share[t, e:e + 1] * _glu(x[t], *p("e%d" % e))
    return y


def _exact_plan(case, seed):
    records, _, args = _plan_records(case)
    tensors, ids, n = _plan_tensors(case, seed), _plan_ids(case, seed), _lengths(case)
    pinepel, ends = case["stack"] == "pinepel", []
    for seq, t in zip(ids, n):
        x, first = tensors[-1, "embed"][seq].double(), None
        for l, m in enumerate(records):
            w = lambda name: tensors[l, name].double()
            if pinepel:
                about = lambda y, name: _rms(y) * (1.0 + w(name))
                y = (_latent if m["mixer"] == xh.MIXER_LATENT else _delta)(about(x, "norm1"), w, m)
                x = x + about(y, "norm1b") * w("ls1")
                x = x + about(_glu(about(x, "norm2"), w("mlp.gate"), w("mlp.up"), w("mlp.down")), "norm2b") * w("ls2")
            else:
                squash = lambda name: torch.tanh(w(name + ".alpha") * x) * w(name) + w(name + ".b")
                y, own = _grouped(squash("norm1"), w, m, first)
                first = own if first is None else first
                x = x + y + _routed(squash("norm2"), w, m)
                side = args["side_dim"]
                e = tensors[-1, "side.embed"][seq][:, l * side:(l + 1) * side].double()
                x = x + _rms((torch.nn.functional.gelu(x @ w("side.gate").T, approximate="tanh") * e) @ w("side.proj").T) * w("side.norm")
        x = x[t - 1:]
        fin = tensors[-1, "final.norm"].double()
        if pinepel:
            ends.append((_rms(x) * (1.0 + fin)) @ tensors[-1, "head"].double().T)
        else:
            z = torch.tanh(tensors[-1, "final.norm.alpha"].double() * x) * fin + tensors[-1, "final.norm.b"].double()
            ends.append(z @ tensors[-1, "embed"].double().T)
    return [torch.stack([e[k] for e in ends]) for k in range(case["new"] + 1)]
