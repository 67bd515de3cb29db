"""GPU parity of the weight path: pack/unpack round trip, bit-exact dequantisation and the
dequant-fused GEMM against the CPU oracle, all through the C-ABI."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KINDS = {"int8": 0, "uint4": 1, "nf4": 2}


@pytest.fixture(scope="module")
def xh():
    from xfastertransformer_amd import capi
    capi.init(0)
    return capi


@pytest.fixture(scope="module")
def orc():
    from oracle import pyoracle
    return pyoracle


def _weights(orc, kind, K, N, seed, asym_int8=False):
    rng = np.random.default_rng(seed)
    W = (rng.standard_normal((K, N)) * 0.02).astype(np.float32)
    w = orc.quantize(kind, W)
    if asym_int8:
        w.zero = (rng.standard_normal(N) * 0.01).astype(np.float32)
    return W, w


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4"])
@pytest.mark.parametrize("K,N", [(256, 64), (4096, 4096), (1000, 250), (11008, 96)])
def test_pack_roundtrip_and_dequant_bit_exact(xh, orc, kind, K, N):
    print(f"case kind={kind} K={K} N={N}", flush=True)
    k = KINDS[kind]
    _, w = _weights(orc, k, K, N, 1, asym_int8=(kind == "int8" and N == 250))
    dw = xh.Weight(k, K, N, w.q, w.scale, w.zero)
    assert np.array_equal(dw.unpack(), w.q)
    assert np.array_equal(dw.dequant(xh.F32).view(np.uint32), orc.dequant(w).view(np.uint32))
    assert np.array_equal(dw.dequant(xh.BF16), orc.dequant_bf16(w))
    dw.free()


def test_gateup_pack_roundtrip(xh, orc):
    K, I = 512, 176
    _, w = _weights(orc, 0, K, 2 * I, 2)
    dw = xh.Weight(0, K, 2 * I, w.q, w.scale, w.zero, flags=xh.WF_GATEUP)
    assert np.array_equal(dw.unpack(), w.q)
    assert np.array_equal(dw.dequant(xh.F32).view(np.uint32), orc.dequant(w).view(np.uint32))


def test_device_quantizer_matches_oracle_definition(xh, orc):
    rng = np.random.default_rng(3)
    W = (rng.standard_normal((384, 96)) * 0.02).astype(np.float32)
    for k in (0, 1, 2):
        q, s, z = xh.quantize_weight(k, W)
        w = orc.quantize(k, W)
        assert np.array_equal(q, w.q) and np.array_equal(s, w.scale)
        if k == 1:
            assert np.array_equal(z, w.zero)


def _run_gemm(xh, dw, A_bits, M, K, N, c_dtype, epi=0, bias=None, res=None, gamma=1.0):
    a_dev = xh.DeviceBuffer.from_numpy(A_bits)
    c_dev = xh.DeviceBuffer(M * N * 4)
    c_dev.zero()
    b_dev = None if bias is None else xh.DeviceBuffer.from_numpy(bias)
    r_dev = None if res is None else xh.DeviceBuffer.from_numpy(res)
    xh.gemm(dw, a_dev.ptr, M, K, c_dev.ptr, N, c_dtype, epi, None if b_dev is None else b_dev.ptr,
            None if r_dev is None else r_dev.ptr, N, xh.F32, gamma)
    xh.synchronize()
    if c_dtype == xh.F32:
        return c_dev.to_numpy(np.float32, (M, N))
    return xh.bf16_bits_to_f32(c_dev.to_numpy(np.uint16, (M, N)))


def _cos(a, b):
    a, b = a.astype(np.float64).ravel(), b.astype(np.float64).ravel()
    return float(a @ b / np.sqrt((a @ a) * (b @ b)))


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4"])
@pytest.mark.parametrize("M", [1, 3, 8, 16, 17, 32])
@pytest.mark.parametrize("K,N", [(4096, 4096), (512, 80), (11008, 256), (4096, 11008)])
def test_skinny_gemm_vs_oracle(xh, orc, kind, M, K, N):
    if (K, N) == (4096, 11008) and M not in (1, 32):
        pytest.skip("large shape covered at M=1 and M=32")
    print(f"case kind={kind} M={M} K={K} N={N}", flush=True)
    k = KINDS[kind]
    _, w = _weights(orc, k, K, N, 10 + M, asym_int8=(kind == "int8" and N == 80))
    rng = np.random.default_rng(100 + M)
    A = orc.round_bf16(rng.standard_normal((M, K)))
    dw = xh.Weight(k, K, N, w.q, w.scale, w.zero)
    got32 = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.F32)
    exp = orc.qgemm(w, A)
    # north-star tolerance on outputs: max-abs 2e-2, cosine >= 0.9999; fp32 output is far inside
    tol = 2e-3
    assert np.abs(got32 - exp).max() < tol, np.abs(got32 - exp).max()
    assert _cos(got32, exp) >= 0.9999
    # bf16 storage adds up to half a bf16 ulp (2^-9 relative) on top
    got16 = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.BF16)
    assert (np.abs(got16 - exp) <= tol + np.abs(exp) * 2.0 ** -8).all()
    assert _cos(got16, exp) >= 0.9999
    dw.free()


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4"])
@pytest.mark.parametrize("M", [33, 64, 200, 256])
@pytest.mark.parametrize("K,N", [(4096, 4096), (512, 80), (1000, 250), (11008, 512)])
def test_mfma_gemm_vs_oracle(xh, orc, kind, M, K, N):
    """M > 32 goes to the MFMA-tiled kernel: same parity bar as the small-M kernel."""
    if (K, N) == (4096, 4096) and M not in (64, 256):
        pytest.skip("large shape covered at M=64 and M=256")
    print(f"case kind={kind} M={M} K={K} N={N}", flush=True)
    k = KINDS[kind]
    _, w = _weights(orc, k, K, N, 50 + M, asym_int8=(kind == "int8" and N == 80))
    rng = np.random.default_rng(150 + M)
    A = orc.round_bf16(rng.standard_normal((M, K)))
    dw = xh.Weight(k, K, N, w.q, w.scale, w.zero)
    got32 = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.F32)
    exp = orc.qgemm(w, A)
    assert np.abs(got32 - exp).max() < 2e-3, np.abs(got32 - exp).max()
    assert _cos(got32, exp) >= 0.9999
    bias = rng.standard_normal(N).astype(np.float32)
    res = rng.standard_normal((M, N)).astype(np.float32)
    got = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.F32, orc.EPI_RESIDENTIAL, bias, res)
    assert np.abs(got - orc.qgemm(w, A, orc.EPI_RESIDENTIAL, bias=bias, res=res)).max() < 2e-3
    dw.free()


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4"])
@pytest.mark.parametrize("M", [40, 256])
def test_mfma_gateup_silu_vs_oracle(xh, orc, kind, M):
    K, I = 1024, 2816
    k = KINDS[kind]
    _, w = _weights(orc, k, K, 2 * I, 60)
    rng = np.random.default_rng(61 + M)
    A = orc.round_bf16(rng.standard_normal((M, K)))
    dw = xh.Weight(k, K, 2 * I, w.q, w.scale, w.zero, flags=xh.WF_GATEUP)
    a_dev = xh.DeviceBuffer.from_numpy(orc.to_bf16(A))
    o_dev = xh.DeviceBuffer(M * I * 4)
    xh.gemm_gateup_silu(dw, a_dev.ptr, M, K, o_dev.ptr, I, xh.F32)
    xh.synchronize()
    got = o_dev.to_numpy(np.float32, (M, I))
    exp = orc.silu_sum(orc.qgemm(w, A))
    assert np.abs(got - exp).max() < 2e-3 + 2e-4 * np.abs(exp).max()
    dw.free()


def _random_weight(xh, orc, rng, kind, K, N, gateup=False):
    """Packed weight, its values in 64 bits and the size of what the kernel adds up (bound below), by code."""
    scale = rng.uniform(0.5e-2, 1.5e-2, N).astype(np.float32)
    flags = xh.WF_GATEUP if gateup else xh.WF_NONE
    if kind == "bf16":
        W = orc.round_bf16(rng.standard_normal((K, N), dtype=np.float32) * 0.05)
        return xh.Weight(xh.W_BF16, K, N, orc.to_bf16(W), flags=flags), W.astype(np.float64), np.abs(W).astype(np.float64)
    if kind.startswith("int8"):
        q = rng.integers(-127, 128, (K, N)).astype(np.int8)
        zero = (rng.standard_normal(N) * 0.05).astype(np.float32) if kind == "int8z" else None
        W = q * scale.astype(np.float64) + (0.0 if zero is None else zero.astype(np.float64))
        return xh.Weight(xh.W_INT8, K, N, q, scale, zero, flags=flags), W, np.abs(q) * scale.astype(np.float64) + (0.0 if zero is None else np.abs(zero))
    u = rng.integers(0, 16, (K, N)).astype(np.uint8)
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).astype(np.uint8)
    if kind == "uint4":
        zero = (-7.5 * scale).astype(np.float32)
        # (the matrix units multiply 128 + code, the row sums take 128 off again)
        return xh.Weight(xh.W_UINT4, K, N, packed, scale, zero, flags=flags), u * scale.astype(np.float64) + zero, (144.0 + u) * scale + np.abs(zero)
    w = xh.Weight(xh.W_NF4, K, N, packed, scale, flags=flags)
    W = w.dequant().astype(np.float64)  # (pinned bit for bit above)
    return w, W, np.abs(W)


# Shapes that between them take every form that any shape takes (test_gemm_forms_host.py checks that they do), with ragged last blocks: 32 and 64
# rows, 128 x 128 and 128 x 256 with one and two K groups, each with K whole and in parts, bands of one to eight row blocks
MANY_ROWS = [(33, 8192, 3088), (97, 4096, 1040), (129, 1024, 12304), (200, 4096, 6160), (450, 11008, 2064), (641, 8192, 4112), (700, 4096, 4112),
             (1285, 4096, 4112), (2100, 1024, 6160), (1161, 2048, 2832), (300, 4160, 2064), (770, 2048, 80),
             # (a depth that is no whole number of 64, whole and broken packed tiles of BF16 weights)
             (2000, 1056, 4112), (1000, 1056, 4112), (300, 8224, 2064), (130, 8224, 2064), (2000, 1064, 4112), (700, 1064, 2064),
             (5526, 12368, 32), (2308, 256, 2512), (2335, 9216, 400), (2129, 12288, 400), (5008, 5248, 160), (2089, 18304, 224), (2307, 3072, 2480),
             (2423, 9216, 784), (1158, 4480, 3296), (1841, 10368, 32),
             # (96 x 256: K in parts, whole, whole for BF16 weights too)
             (66, 4096, 12944), (652, 512, 11040), (579, 512, 12912), (1155, 512, 6720)]


@pytest.mark.parametrize("kind", ["int8", "int8z", "uint4", "nf4", "bf16"])
@pytest.mark.parametrize("M,K,N", MANY_ROWS)
def test_mfma_every_tile_against_64_bits(xh, orc, kind, M, K, N):
    """Bound: K + 8 additions and the epilogue's few operations in fp32, each off by 2^-24 of what has been added up so far at most; NF4 values
    go in as two bf16 parts, off by 2^-17."""
    rng = np.random.default_rng(M + K + N)
    w, W, size = _random_weight(xh, orc, rng, kind, K, N)
    A = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32))
    got = _run_gemm(xh, w, orc.to_bf16(A), M, K, N, xh.F32)
    bound = np.abs(A).astype(np.float64) @ size * ((K + 8) * 2.0 ** -24 + (2.0 ** -16 if kind == "nf4" else 0.0))
    worst = float((np.abs(got - A.astype(np.float64) @ W) / bound).max())
    print(f"case {kind} {M} x {N} x {K}: {worst:.2e} of the bound", flush=True)
    assert worst <= 1.0
    w.free()


# on 256 CUs: 1, 2, 3, 4 (at 17 rows and more) and 6 column tiles a block, ragged last blocks, 8 to 1 K slices, and more than 8 tiles a CU
FEW_ROWS = [(M, K, N) for K, N in [(1280, 1040), (1280, 4112), (1280, 9232), (768, 13328), (768, 18448), (768, 28672), (768, 36880), (256, 36880)]
            for M in (3, 13, 29)] + [(13, 4096, 1040), (13, 256, 49200)]


@pytest.mark.parametrize("kind", ["int8", "int8z", "uint4", "nf4", "bf16"])
@pytest.mark.parametrize("M,K,N", FEW_ROWS)
def test_few_rows_every_form_against_64_bits(xh, orc, kind, M, K, N):
    test_mfma_every_tile_against_64_bits(xh, orc, kind, M, K, N)


@pytest.mark.parametrize("kind", ["uint4", "nf4"])
@pytest.mark.parametrize("M,K,N", [(5, 128, 48), (16, 384, 80), (17, 128, 4112), (31, 256, 12304), (32, 1152, 2064), (17, 4352, 16), (32, 640, 20496), (16, 128, 49168), (16, 384, 49152),
                                   (24, 640, 37904), (32, 1152, 18944)])
def test_rows_straight_into_lds_against_64_bits(xh, orc, kind, M, K, N):
    """One load batch a slice, an odd number and unequal ones; rows that fill their 16-row tiles and a single one in the second."""
    test_mfma_every_tile_against_64_bits(xh, orc, kind, M, K, N)


@pytest.mark.parametrize("kind", ["uint4", "nf4"])
def test_rows_four_gigabytes_apart(xh, orc, kind):
    """The last row begins beyond the reach of 32-bit byte offsets."""
    M, K, N, lda = 17, 256, 48, 134217728
    rng = np.random.default_rng(3)
    w, W, size = _random_weight(xh, orc, rng, kind, K, N)
    A = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32))
    a_dev, o_dev = xh.DeviceBuffer(((M - 1) * lda + K) * 2), xh.DeviceBuffer(M * N * 4)
    for m in range(M):
        a_dev.upload(orc.to_bf16(A[m]), m * lda * 2)
    xh.gemm(w, a_dev.ptr, M, lda, o_dev.ptr, N, xh.F32)
    xh.synchronize()
    bound = np.abs(A).astype(np.float64) @ size * ((K + 8) * 2.0 ** -24 + (2.0 ** -16 if kind == "nf4" else 0.0))
    assert float((np.abs(o_dev.to_numpy(np.float32, (M, N)) - A.astype(np.float64) @ W) / bound).max()) <= 1.0
    a_dev.free()
    w.free()


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4", "bf16"])
@pytest.mark.parametrize("M,lda,gateup", [
    (17, 120000000, 0),  # the last rows behind 2 GB, within reach of unsigned byte offsets
    (40, 50000000, 0),
    (17, 1 << 28, 0),  # a row 2^32 elements behind the first
    (33, 1 << 27, 1),
    (70, 1 << 26, 0),  # (and a product of six rows for the rest)
])
def test_rows_gigabytes_apart(xh, orc, kind, M, lda, gateup):
    """Few and many rows whose places 32-bit offsets hold, of bytes or of elements, and those that they do not; with the residual, which has rows of its own."""
    K, N = 256, 64
    rng = np.random.default_rng(M)
    w, W, size = _random_weight(xh, orc, rng, kind, K, N, gateup=bool(gateup))
    A, R = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32)), rng.standard_normal((M, N), dtype=np.float32)
    a_dev, r_dev, o_dev = xh.DeviceBuffer(((M - 1) * lda + K) * 2), xh.DeviceBuffer.from_numpy(R), xh.DeviceBuffer(M * N * 4)
    for m in range(M):
        a_dev.upload(orc.to_bf16(A[m]), m * lda * 2)
    if gateup:
        xh.gemm_gateup_silu(w, a_dev.ptr, M, lda, o_dev.ptr, N // 2, xh.F32)
    else:
        xh.gemm(w, a_dev.ptr, M, lda, o_dev.ptr, N, xh.F32, xh.EPI_RESIDENTIAL, res=r_dev.ptr, ldres=N)
    xh.synchronize()
    got = o_dev.to_numpy(np.float32, (M, N // 2 if gateup else N))
    y, b = A.astype(np.float64) @ W, np.abs(A).astype(np.float64) @ size * ((K + 8) * 2.0 ** -24 + (2.0 ** -16 if kind == "nf4" else 0.0))
    if gateup:  # (the bound of test_mfma_gateup_every_tile_against_64_bits)
        g, u = y[:, :N // 2], y[:, N // 2:]
        silu = g / (1.0 + np.exp(-g))
        want, bound = silu * u, 1.1 * b[:, :N // 2] * np.abs(u) + b[:, N // 2:] * (np.abs(silu) + 1.1 * b[:, :N // 2]) + np.abs(silu * u) * 2.0 ** -20
    else:
        want, bound = y + R, b + np.abs(y + R) * 2.0 ** -23
    assert float((np.abs(got - want) / bound).max()) <= 1.0
    a_dev.free()
    w.free()


@pytest.mark.parametrize("M", [4, 5, 16])
@pytest.mark.parametrize("K,N", [(3968, 40), (4096, 40), (4224, 16), (4480, 4096), (5632, 2048)])
def test_bf16_tiles_alone_on_their_cu_against_64_bits(xh, orc, M, K, N):
    """The shallowest K of the form and one below it; slices of as many load batches, of one more and of an odd number (the last sum's)."""
    test_mfma_every_tile_against_64_bits(xh, orc, "bf16", M, K, N)


GATE_UP = [(3, 768, 1040), (13, 768, 14336), (29, 768, 9232), (29, 768, 18448), (100, 1024, 1040), (700, 2048, 2064), (1285, 4096, 2064), (2100, 1024, 3088),
           (23, 128, 16), (2, 128, 17392), (12, 128, 17408), (1966, 13312, 1280)]


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4", "bf16"])
@pytest.mark.parametrize("M,K,I", GATE_UP)
def test_mfma_gateup_every_tile_against_64_bits(xh, orc, kind, M, K, I):
    """silu(g) u: off by what the bounds of g and u (test above) make of it, |silu'| <= 1.1, and 2^-20 of the value for the exponential."""
    rng = np.random.default_rng(M + I)
    w, W, size = _random_weight(xh, orc, rng, kind, K, 2 * I, gateup=True)
    A = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32))
    a_dev, o_dev = xh.DeviceBuffer.from_numpy(orc.to_bf16(A)), xh.DeviceBuffer(M * I * 4)
    xh.gemm_gateup_silu(w, a_dev.ptr, M, K, o_dev.ptr, I, xh.F32)
    xh.synchronize()
    got = o_dev.to_numpy(np.float32, (M, I))
    y, b = A.astype(np.float64) @ W, np.abs(A).astype(np.float64) @ size * ((K + 8) * 2.0 ** -24 + (2.0 ** -16 if kind == "nf4" else 0.0))
    g, u = y[:, :I], y[:, I:]
    silu = g / (1.0 + np.exp(-g))
    bound = 1.1 * b[:, :I] * np.abs(u) + b[:, I:] * (np.abs(silu) + 1.1 * b[:, :I]) + np.abs(silu * u) * 2.0 ** -20
    assert float((np.abs(got - silu * u) / bound).max()) <= 1.0
    w.free()


def test_bf16_weight_gemm_both_kernels(xh, orc):
    rng = np.random.default_rng(70)
    K, N = 512, 1000
    W = orc.round_bf16(rng.standard_normal((K, N)) * 0.05)
    dw = xh.Weight(xh.W_BF16, K, N, orc.to_bf16(W))
    assert np.array_equal(dw.unpack(), orc.to_bf16(W))
    for M in (3, 77):
        A = orc.round_bf16(rng.standard_normal((M, K)))
        got = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.F32)
        assert np.abs(got - orc.gemm_f32(A, W)).max() < 1e-3


@pytest.mark.parametrize("epi", ["bias", "silu", "gelu", "resmul", "residential", "residential_bias", "resext"])
def test_skinny_gemm_epilogues(xh, orc, epi):
    M, K, N = 5, 1024, 272
    _, w = _weights(orc, 0, K, N, 20)
    rng = np.random.default_rng(21)
    A = orc.round_bf16(rng.standard_normal((M, K)))
    bias = rng.standard_normal(N).astype(np.float32)
    res = rng.standard_normal((M, N)).astype(np.float32)
    dw = xh.Weight(0, K, N, w.q, w.scale, w.zero)
    table = {"bias": (orc.EPI_BIAS, bias, None), "silu": (orc.EPI_SILU, None, None),
             "gelu": (orc.EPI_GELU, None, None), "resmul": (orc.EPI_RESMUL, None, res),
             "residential": (orc.EPI_RESIDENTIAL, None, res), "residential_bias": (orc.EPI_RESIDENTIAL, bias, res),
             "resext": (orc.EPI_RESEXT, None, res)}
    e, b, r = table[epi]
    exp = orc.qgemm(w, A, e, bias=b, res=r, gamma=0.5)
    got = _run_gemm(xh, dw, orc.to_bf16(A), M, K, N, xh.F32, e, b, r, 0.5)
    assert np.abs(got - exp).max() < 2e-3


@pytest.mark.parametrize("kind", ["int8", "uint4", "nf4"])
@pytest.mark.parametrize("M", [1, 8, 32])
def test_gateup_silu_vs_oracle(xh, orc, kind, M):
    K, I = 4096, 11008
    k = KINDS[kind]
    _, w = _weights(orc, k, K, 2 * I, 30)
    rng = np.random.default_rng(31 + M)
    A = orc.round_bf16(rng.standard_normal((M, K)))
    dw = xh.Weight(k, K, 2 * I, w.q, w.scale, w.zero, flags=xh.WF_GATEUP)
    a_dev = xh.DeviceBuffer.from_numpy(orc.to_bf16(A))
    o_dev = xh.DeviceBuffer(M * I * 4)
    xh.gemm_gateup_silu(dw, a_dev.ptr, M, K, o_dev.ptr, I, xh.F32)
    xh.synchronize()
    got = o_dev.to_numpy(np.float32, (M, I))
    exp = orc.silu_sum(orc.qgemm(w, A))
    assert np.abs(got - exp).max() < 2e-3 + 2e-4 * np.abs(exp).max()
    assert _cos(got, exp) >= 0.9999
    dw.free()


def test_gemm_rejects_bad_arguments(xh, orc):
    _, w = _weights(orc, 0, 256, 64, 40)
    dw = xh.Weight(0, 256, 64, w.q, w.scale, w.zero)
    a = xh.DeviceBuffer(32 * 256 * 2)
    c = xh.DeviceBuffer(32 * 64 * 4)
    with pytest.raises(xh.XftHipError):
        xh.gemm(dw, a.ptr, 1, 100, c.ptr, 64)  # lda < K
    with pytest.raises(xh.XftHipError):
        xh.gemm(dw, a.ptr, 1, 256, c.ptr, 32)  # ldc < N
    with pytest.raises(xh.XftHipError):
        xh.gemm(dw, a.ptr, 1, 256, c.ptr, 64, epi=xh.EPI_BIAS)  # bias missing
    with pytest.raises(xh.XftHipError):
        xh.gemm_gateup_silu(dw, a.ptr, 1, 256, c.ptr, 32)  # not a gate/up weight


@pytest.mark.parametrize("kind", ["int8", "bf16"])
def test_null_stream_beside_a_capture(xh, orc, kind):
    """A product whose K is split, on the null stream, while another stream is being captured: the bits of an ordinary call."""
    import ctypes as C
    M, K, N = 64, 4096, 1024
    rng = np.random.default_rng(4)
    w, _, _ = _random_weight(xh, orc, rng, kind, K, N)
    a = orc.to_bf16(orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32)))
    want = _run_gemm(xh, w, a, M, K, N, xh.F32)
    a_dev, c_dev, stream, graph = xh.DeviceBuffer.from_numpy(a), xh.DeviceBuffer(M * N * 4), xh.Stream(), C.c_void_p()
    assert xh.lib.hipStreamBeginCapture(stream.h, 1) == 0  # 1: thread-local checks
    try:
        xh.gemm(w, a_dev.ptr, M, K, c_dev.ptr, N, xh.F32)
    finally:
        assert xh.lib.hipStreamEndCapture(stream.h, C.byref(graph)) == 0
        xh.lib.hipGraphDestroy(graph)
    xh.synchronize()
    assert np.array_equal(c_dev.to_numpy(np.float32, (M, N)), want)
    w.free()


@pytest.mark.parametrize("kind", ["int8", "int8z", "uint4", "nf4", "bf16"])
@pytest.mark.parametrize("M,K,N", [(33, 8192, 3088), (200, 4096, 6160), (700, 4096, 4112), (641, 8192, 4112), (2308, 256, 2512), (2335, 9216, 400), (2129, 12288, 400),
                                   (2100, 1024, 6160), (2000, 1056, 4112), (13, 768, 13328), (29, 768, 28672), (3, 768, 36880)])
def test_epilogues_of_the_forms_against_64_bits(xh, orc, kind, M, K, N):
    """Bias and residual on top of the sums, and bf16 results: the bound of the product, three more roundings of 2^-24 of the terms, and half a step
    of the bf16 result (8 significant bits: 2^-8 of it at most)."""
    rng = np.random.default_rng(M + K + N)
    w, W, size = _random_weight(xh, orc, rng, kind, K, N)
    A = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32))
    bias, res = rng.standard_normal(N).astype(np.float32), rng.standard_normal((M, N)).astype(np.float32)
    y = A.astype(np.float64) @ W
    bound = np.abs(A).astype(np.float64) @ size * ((K + 8) * 2.0 ** -24 + (2.0 ** -16 if kind == "nf4" else 0.0))
    got = _run_gemm(xh, w, orc.to_bf16(A), M, K, N, xh.F32, xh.EPI_RESIDENTIAL, bias, res)
    assert (np.abs(got - (y + bias + res)) <= bound + 3 * 2.0 ** -24 * (np.abs(y) + np.abs(bias) + np.abs(res))).all()
    got = _run_gemm(xh, w, orc.to_bf16(A), M, K, N, xh.BF16)
    assert (np.abs(got - y) <= bound * (1 + 2.0 ** -8) + np.abs(y) * 2.0 ** -8).all()
    w.free()


@pytest.mark.parametrize("kind", ["int8", "uint4", "bf16"])
def test_captured_without_a_parts_buffer(xh, orc, kind):
    """A product whose K is split, captured on a stream that has no buffer for the parts, runs unsplit: within the bound of the product, the
    same bits on every replay (not those of the split form, whose sums have another order)."""
    import ctypes as C
    M, K, N = 64, 4096, 1024
    rng = np.random.default_rng(6)
    w, W, size = _random_weight(xh, orc, rng, kind, K, N)
    assert xh.gemm_form({"int8": xh.W_INT8, "uint4": xh.W_UINT4, "bf16": xh.W_BF16}[kind], M, K, N, has_zero=kind == "uint4")[3] > 1
    A = orc.round_bf16(rng.standard_normal((M, K), dtype=np.float32))
    a, out, graph = xh.DeviceBuffer.from_numpy(orc.to_bf16(A)), xh.DeviceBuffer(M * N * 4), C.c_void_p()
    _unused.append(xh.Stream())
    stream = _unused[-1]
    assert xh.lib.hipStreamBeginCapture(stream.h, 1) == 0  # as another library would; 1: thread-local checks
    xh.gemm(w, a.ptr, M, K, out.ptr, N, xh.F32, stream=stream.h)
    assert xh.lib.xfthip_graph_end(stream.h, C.byref(graph)) == 0
    bound, first = np.abs(A).astype(np.float64) @ size * (K + 8) * 2.0 ** -24, None
    for _ in range(3):
        out.zero()
        assert xh.lib.xfthip_graph_launch(graph, stream.h) == 0
        xh.synchronize()
        got = out.to_numpy(np.float32, (M, N))
        assert (np.abs(got - A.astype(np.float64) @ W) <= bound).all()
        first = got if first is None else first
        assert np.array_equal(got, first)
    xh.lib.xfthip_graph_destroy(graph)
    w.free()


_unused = []  # streams kept alive: scratch is kept by a stream's handle, which a destroyed one's successor may get


@pytest.mark.parametrize("M", [1, 4, 5, 16])
def test_ragged_k_in_one_sum(xh, M):
    """BF16 weights, K no multiple of the 32-row weight tile: what cancels in the first two tiles leaves the third's as it is.  In two sums in turn, the third
    tile's 1 is lost beside the first's 2^24."""
    K, N = 232, 48
    A, W = np.zeros((M, K), np.float32), np.zeros((K, N), np.float32)
    A[:, [3, 35, 70]], W[3], W[35], W[70] = [4096.0, 4096.0, 1.0], 4096.0, -4096.0, 1.0
    dw = xh.Weight(xh.W_BF16, K, N, xh.f32_to_bf16_bits(W))
    assert (_run_gemm(xh, dw, xh.f32_to_bf16_bits(A), M, K, N, xh.F32) == 1.0).all()
    dw.free()


@pytest.mark.parametrize("kind", ["uint4", "nf4"])
@pytest.mark.parametrize("M,K,N,direct", [(2100, 192, 6160, 1), (2308, 320, 2512, 1), (2000, 1088, 4112, 1), (2129, 12352, 400, 1), (2100, 64, 6160, 0)])
def test_four_bit_steps_of_half_a_tile_against_64_bits(xh, orc, kind, M, K, N, direct):
    """4-bit weights, K an odd number of 64: the last step of the tiles with activations straight into LDS is half a packed tile (the last shape is another tile's)."""
    assert xh.gemm_form({"uint4": xh.W_UINT4, "nf4": xh.W_NF4}[kind], M, K, N, 0, kind == "uint4")[4] == direct
    test_mfma_every_tile_against_64_bits(xh, orc, kind, M, K, N)


@pytest.mark.parametrize("kind,M,N,tile", [("uint4", 773, 18000, (128, 256)), ("uint4", 810, 14000, (96, 256)), ("nf4", 1437, 8192, (96, 256)), ("nf4", 3585, 10800, (128, 128))])
def test_half_a_packed_tile_alone_against_64_bits(xh, orc, kind, M, N, tile):
    """4-bit weights, K = 64: the only step of the tiles with activations straight into LDS is half a packed tile, in front of which there is nothing to request."""
    assert xh.gemm_form({"uint4": xh.W_UINT4, "nf4": xh.W_NF4}[kind], M, 64, N, 0, kind == "uint4") == tile + (1, 1, 1)
    test_mfma_every_tile_against_64_bits(xh, orc, kind, M, 64, N)
