"""The packed preparation's float16 division, on the CPU (no GPU needed)."""

from __future__ import annotations

import ctypes

import numpy as np


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
