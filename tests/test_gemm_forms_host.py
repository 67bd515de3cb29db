"""The shapes of the GPU tests of the products take every form of the kernels that any shape takes: which form a product takes is decided on the
host and needs no device."""
import os
import random
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import test_qgemm_gpu as gpu  # noqa: E402

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "xfastertransformer_amd")
pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(PKG, "libxft_hip.so")), reason="library not built (run __graft_entry__.build())")


@pytest.fixture(scope="module")
def xh():
    from xfastertransformer_amd import capi
    return capi


def _form(xh, kind, M, K, N, gateup=False):
    """What tells one built kernel from another, and whether K goes in parts."""
    code, zero = {"int8": (xh.W_INT8, False), "int8z": (xh.W_INT8, True), "uint4": (xh.W_UINT4, True), "nf4": (xh.W_NF4, False),
                  "bf16": (xh.W_BF16, False)}[kind]
    f = xh.gemm_form(code, M, K, N, xh.WF_GATEUP if gateup else 0, zero)
    if M <= 32:
        return (M + 15) // 16, M > 4, f[0], f[1]
    rows, cols, groups, parts, direct = f
    return rows, cols, groups, direct, parts > 1, K % (32 if kind == "bf16" else 64) != 0


@pytest.mark.parametrize("kind", ["int8", "int8z", "uint4", "nf4", "bf16"])
def test_every_form_is_tested(xh, kind):
    rng, reached = random.Random(5), {}
    for _ in range(30000):
        M, gateup = int(2 ** rng.uniform(0, 12.5)), rng.random() < 0.3 and kind != "int8z"
        K = int(2 ** rng.uniform(7, 14.2))
        K = K // 8 * 8 if M > 32 and rng.random() < 0.3 else max(128, K // 128 * 128)
        N = max(32, int(2 ** rng.uniform(5, 17.3)) // 32 * 32)
        reached.setdefault(_form(xh, kind, M, K, N, gateup), (M, K, N, gateup))
    tested = {_form(xh, kind, M, K, N) for M, K, N in gpu.MANY_ROWS + gpu.FEW_ROWS}
    if kind != "int8z":
        tested |= {_form(xh, kind, M, K, 2 * I, True) for M, K, I in gpu.GATE_UP}
    missing = {f: shape for f, shape in reached.items() if f not in tested}
    assert len(reached) > 15 and not missing


def test_staged_tiles_of_a_ragged_depth(xh):
    """K no whole number of 64: 128-row tiles through registers wherever they fill the device, BF16 weights whole packed tiles in 128 x 128 as well."""
    assert xh.gemm_form(xh.W_BF16, 2048, 11040, 4096) == (128, 256, 1, 1, 0)
    assert xh.gemm_form(xh.W_BF16, 1024, 11040, 4096) == (128, 128, 1, 1, 0)
    assert xh.gemm_form(xh.W_INT8, 2048, 11040, 4096) == (128, 256, 1, 1, 0)
    assert xh.gemm_form(xh.W_INT8, 450, 11040, 4096) == (64, 128, 1, 2, 0)


def test_few_rows_of_a_wide_weight(xh):
    """Shallow and deep K over many columns, and a stretch of columns that leaves a CU four blocks of two tiles."""
    assert xh.gemm_form(xh.W_INT8, 8, 2048, 151936)[:3] == (2, 2, 3)
    assert xh.gemm_form(xh.W_BF16, 8, 2048, 151936)[:3] == (2, 2, 3)
    assert xh.gemm_form(xh.W_INT8, 8, 8192, 55296)[:3] == (2, 2, 1)
    assert xh.gemm_form(xh.W_BF16, 32, 1024, 65024)[:3] == (2, 2, 2)
    assert xh.gemm_form(xh.W_BF16, 32, 8192, 28672)[:3] == (2, 2, 1)
    assert xh.gemm_form(xh.W_INT8, 32, 5120, 27648)[:3] == (4, 1, 4)


@pytest.mark.parametrize("M,K,N,form", [(16, 4096, 2048, (1, 4, 4)), (13, 4096, 512, (1, 4, 4)), (12, 4096, 512, (1, 2, 8)), (8, 5632, 2048, (1, 2, 8)), (16, 4128, 4096, (1, 2, 8)),
                                        (16, 3968, 4096, (1, 2, 8)), (7, 4096, 4096, (1, 4, 4)), (7, 11008, 4096, (1, 4, 4)), (7, 8192, 3072, (1, 4, 4)), (6, 11008, 4096, (1, 2, 8)),
                                        (8, 4480, 4096, (1, 2, 8)), (8, 8192, 3056, (1, 2, 8)), (5, 32768, 64, (1, 2, 8))])
def test_bf16_tiles_alone_on_their_cu(xh, M, K, N, form):
    """Four slices of four k tiles where they gain (256 CUs): many rows, or most CUs at work over slices of whole pairs of batches; eight of two elsewhere."""
    assert xh.gemm_form(xh.W_BF16, M, K, N)[:3] == form
