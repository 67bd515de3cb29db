"""Narrowing to bf16 on the device: results that leave the products in bf16 have the bits of the reference's conversion."""
import os
import subprocess

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _patterns():
    """fp32 bit patterns about every border of the conversion: all exponents, mantissas about the rounding borders, both signs, NaN with payloads."""
    low = np.asarray([0, 1, 0x7FFF, 0x8000, 0x8001, 0xFFFF, 0x10000, 0x17FFF, 0x18000, 0x18001, 0x3F8000, 0x400000, 0x7F7FFF, 0x7F8000, 0x7FFFFF], np.uint32)
    u = ((np.arange(256, dtype=np.uint32) << 23)[:, None] | low[None, :]).ravel()
    u = u[u != 0]  # (zero plus minus zero is zero)
    return np.concatenate([u, u | np.uint32(0x80000000)])


@pytest.mark.parametrize("M", [3, 48, 320])
def test_every_class_of_value(M):
    """A product of zeros plus a residual: the residual narrowed.  3 rows: one value at a time; 48: chunks of eight; 320: the same from 128-row tiles."""
    from oracle import pyoracle as orc
    from xfastertransformer_amd import capi as xh
    xh.init(0)
    K, N, u = 128, 512, _patterns()
    bits = np.resize(u, M * N).reshape(M, N)
    w = xh.Weight(xh.W_BF16, K, N, np.zeros((K, N), np.uint16))
    for at in range(0, len(u), M * N):
        bits = np.resize(np.roll(u, -at), M * N).reshape(M, N)
        a, res, out = xh.DeviceBuffer.from_numpy(np.zeros((M, K), np.uint16)), xh.DeviceBuffer.from_numpy(bits.view(np.float32)), xh.DeviceBuffer(M * N * 2)
        xh.gemm(w, a.ptr, M, K, out.ptr, N, xh.BF16, orc.EPI_RESIDENTIAL, None, res.ptr, N, xh.F32, 1.0)
        xh.synchronize()
        quiet = np.where((bits & 0x7FFFFFFF) > 0x7F800000, bits | 0x400000, bits)  # (the sum quiets a signalling NaN)
        assert np.array_equal(out.to_numpy(np.uint16, (M, N)), orc.to_bf16(quiet.view(np.float32)))
    w.free()


def test_all_patterns():
    """The conversion that every kernel compiles, over all 2^32 bit patterns in both halves of a pair."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    sweep = os.path.join(root, "xfastertransformer_amd", "csrc", "build", "bf16_device_sweep")
    assert os.path.exists(sweep), "tests/bf16_device_sweep.hip is not built; run `python -m xfastertransformer_amd.build`"
    out = subprocess.run([sweep], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0 and out.stdout == "mismatches lo=0 hi=0 one=0\n", out.stdout + out.stderr
