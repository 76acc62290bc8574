"""The few-row linear's argument checks and ConvRotLinear's rule for it (no GPU needed)."""

from __future__ import annotations

import pytest
import torch

from convrot_mlx_amd import _native as nat
from convrot_mlx_amd import core


def _call(x=4096, dtype=nat.DTYPE_BF16, group=64, a4=1, w=1 << 20, ws=1 << 21, bias=None, M=1, N=64, K=1024,
          residual=None, gate=None, stride=0, rpg=1, out=1 << 22):
    return nat.load().convrot_linear_rows(x, dtype, group, a4, w, ws, bias, M, N, K, residual, gate, stride, rpg, out,
                                          None)


@pytest.mark.parametrize("bad,status", [
    ({"dtype": 7}, nat.ERR_INVALID), ({"M": -1}, nat.ERR_INVALID), ({"group": 96}, nat.ERR_INVALID),
    ({"K": 1056}, nat.ERR_INVALID), ({"gate": 4096}, nat.ERR_INVALID),
    ({"residual": 4096, "gate": 4096, "rpg": 0}, nat.ERR_INVALID),
    ({"x": None}, nat.ERR_INVALID), ({"out": 8}, nat.ERR_INVALID), ({"residual": 8}, nat.ERR_INVALID),
    ({"x": 4096, "out": 4096 + 2032}, nat.ERR_INVALID), ({"x": 4096, "out": 4096 - 112}, nat.ERR_INVALID),
    ({"group": 16}, nat.ERR_UNSUPPORTED), ({"group": 1024}, nat.ERR_UNSUPPORTED), ({"M": 17}, nat.ERR_UNSUPPORTED),
    ({"M": 9, "K": 2048}, nat.ERR_UNSUPPORTED), ({"a4": 0, "dtype": nat.DTYPE_F32}, nat.ERR_UNSUPPORTED),
    ({"N": 1 << 30, "K": 8192}, nat.ERR_UNSUPPORTED),
])
def test_refusals(bad, status):
    """Null, misaligned and overlapping buffers and shapes outside the kernel's are refused before any launch."""
    assert _call(**bad) == status
    assert nat.load().convrot_last_error()


def test_empty_products():
    assert _call(M=0) == nat.OK and _call(N=0) == nat.OK


@pytest.mark.parametrize("rows,k,dtype,group,a4,takes", [
    (1, 16384, torch.bfloat16, 256, True, True), (1, 16640, torch.bfloat16, 256, True, False),
    (1, 16384, torch.float32, 256, True, False), (1, 8192, torch.float32, 64, True, True),
    (2, 3072, torch.bfloat16, 64, True, True), (3, 3072, torch.bfloat16, 64, True, False),
    (4, 1536, torch.float16, 64, True, True), (5, 1024, torch.bfloat16, 64, True, False),
    (4, 3072, torch.bfloat16, 64, False, True), (9, 1024, torch.bfloat16, 64, False, False),
    (1, 1024, torch.float32, 64, False, False), (1, 1024, torch.bfloat16, 16, True, False),
    (0, 1024, torch.bfloat16, 64, True, False),
])
def test_rule(rows, k, dtype, group, a4, takes):
    x = torch.empty((rows, k), dtype=dtype, device="meta")
    assert core._linear_rows_eligible(x, group, a4) is takes
