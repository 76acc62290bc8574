"""The packed preparation's float16 division, on the CPU (no GPU needed)."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest

from convrot_mlx_amd import _native as nat


def test_f16_quotient_is_the_division():
    """q = v * (1/s), corrected once by fma(fma(-q, s, v), 1/s, q), rounds to the float16 that the float32
    division v / s rounds to: every pair of float16 significands (a power of two scales every step
    exactly; quotients of the format's denormals are codes 0 either way)."""
    fmaf = ctypes.CDLL("libm.so.6").fmaf
    fmaf.restype, fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    sig = np.arange(1024, 2048, dtype=np.float32)
    for s in sig:
        inv = np.float32(1.0) / s
        want = (sig / s).astype(np.float16)
        q = sig * inv
        # exact in float64: 24 x 11 bits and a subtraction of values a few ulps apart
        e = (sig.astype(np.float64) - q.astype(np.float64) * np.float64(s)).astype(np.float32)
        got = np.array([fmaf(float(a), float(inv), float(b)) if a else b for a, b in zip(e, q)], dtype=np.float32)
        assert np.array_equal(got.astype(np.float16), want), s


BF16, F16, F32 = nat.DTYPE_BF16, nat.DTYPE_F16, nat.DTYPE_F32
PLAIN, MODULATE, GELU = nat.PRODUCER_PLAIN, nat.PRODUCER_MODULATE, nat.PRODUCER_GELU
FP6, INT8, PACKED, ROTATE = nat.PREP_FP6, nat.PREP_INT8, nat.PREP_PACKED, nat.PREP_ROTATE


@pytest.mark.parametrize("rows,k,dtype,group,mode,producer,want", [
    # the kernel of packed values, but for the rows whose FP6 stores or spills made it the slower one
    (4608, 3072, BF16, 256, FP6, PLAIN, (3, 1, True)), (8800, 16384, BF16, 256, FP6, PLAIN, (4, 4, True)),
    (8800, 16384, BF16, 64, FP6, PLAIN, (4, 4, False)), (8800, 8192, BF16, 64, FP6, PLAIN, (1, 8, True)),
    (8800, 12288, BF16, 64, FP6, PLAIN, (3, 4, True)), (4877, 29568, BF16, 64, FP6, PLAIN, (3, 10, True)),
    (1536, 16384, BF16, 64, FP6, PLAIN, (4, 4, True)), (2049, 16384, BF16, 64, FP6, PLAIN, (4, 4, False)),
    (8800, 8192, BF16, 16, FP6, PLAIN, (4, 2, False)), (7020, 1152, BF16, 16, FP6, PLAIN, (1, 2, True)),
    (381, 12288, BF16, 16, FP6, PLAIN, (1, 12, True)), (2000, 12288, BF16, 16, FP6, PLAIN, (1, 12, False)),
    (1061, 14336, BF16, 4, PACKED, PLAIN, (1, 14, False)), (4608, 3072, BF16, 64, ROTATE, PLAIN, (3, 1, False)),
    (4608, 3072, F32, 64, FP6, PLAIN, (3, 1, False)), (8800, 16384, F16, 16, FP6, PLAIN, (1, 16, True)),
    (8800, 16384, F16, 64, FP6, PLAIN, (4, 4, True)),
    # float16 rotated outputs on one iteration
    (2000, 12288, F16, 64, ROTATE, PLAIN, (1, 12, False)), (710, 14336, F16, 64, ROTATE, PLAIN, (1, 14, True)),
    (2048, 10240, F16, 64, ROTATE, PLAIN, (1, 10, True)), (2000, 12288, F16, 256, ROTATE, PLAIN, (1, 12, True)),
    (5879, 7168, F16, 16, ROTATE, MODULATE, (1, 7, False)), (4608, 15360, F16, 16, ROTATE, MODULATE, (4, 4, True)),
    # few rows of many blocks, and thirteen blocks
    (1536, 15360, BF16, 64, INT8, PLAIN, (4, 4, True)), (1536, 15360, BF16, 64, INT8, GELU, (1, 15, True)),
    (1536, 15360, BF16, 64, INT8, MODULATE, (4, 4, False)), (1667, 8192, BF16, 64, INT8, MODULATE, (1, 8, True)),
    (1024, 12288, BF16, 64, INT8, PLAIN, (1, 12, True)), (1025, 12288, BF16, 64, INT8, PLAIN, (3, 4, True)),
    (1536, 12288, BF16, 16, INT8, PLAIN, (1, 12, True)), (4608, 13312, BF16, 256, FP6, PLAIN, (4, 4, True)),
])
def test_route(rows, k, dtype, group, mode, producer, want):
    """(iterations a wave, waves, packed kernel) on each side of the lines of the plan."""
    assert nat.prepare_plan(rows, k, dtype, group, mode, producer) == want


@pytest.mark.parametrize("bad", [dict(rows=-1), dict(k=0), dict(k=65537), dict(dtype=7), dict(group=48), dict(group=4096),
                                 dict(mode=5), dict(producer=3)])
def test_route_refuses(bad):
    args = {"rows": 16, "k": 1024, "dtype": BF16, "group": 64, "mode": INT8, "producer": PLAIN, **bad}
    with pytest.raises(ValueError, match="preparation plan query"):
        nat.prepare_plan(*args.values())
