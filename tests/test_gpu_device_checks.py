"""GPU: arithmetic that the preparation kernels take as exact, over its whole range (tests/device_checks.hip,
built with the library)."""

from __future__ import annotations

import ctypes
from pathlib import Path

import pytest
import torch

pytestmark = pytest.mark.gpu

LIB = Path(__file__).resolve().parent / "libdevice_checks.so"


def _count(dev, name, *args):
    """(disagreements, missed non-finite results, the least input of either, inputs compared) of a check."""
    result = torch.zeros(4, dtype=torch.int64, device=dev)
    result[2] = 2 ** 62
    fn = getattr(ctypes.CDLL(str(LIB)), name)
    fn.argtypes = [ctypes.c_int] * len(args) + [ctypes.c_void_p, ctypes.c_void_p]
    assert fn(*args, result.data_ptr(), torch.cuda.current_stream(dev).cuda_stream) == 0
    return result.tolist()


def test_reciprocal(dev):
    """The GELU's reciprocal is 1 / d rounded, for every float32 d in [1, 2^126)."""
    bad, _, first, compared = _count(dev, "check_reciprocal")
    assert compared == 126 * 2 ** 23
    assert bad == 0, f"{bad} reciprocals differ, the first at {first:#x}"


@pytest.mark.parametrize("regs", [0, 1])
@pytest.mark.parametrize("bf16", [1, 0])
def test_butterflies(dev, bf16, regs):
    """The packed radix-4s are the float32 ones on all 2^32 pairs of values in any two of the four places, the
    other two zero or of like magnitude; results that are not finite are never missed."""
    bad, missed, first, compared = _count(dev, "check_butterflies", bf16, regs)
    assert (bad, missed) == (0, 0), f"first at pair {first:#x}"
    # twelve walks of all pairs: those with an infinity, NaN or overflow in any butterfly are not compared
    assert 12 * 2 ** 32 * (0.95 if bf16 else 0.75) < compared < 12 * 2 ** 32
