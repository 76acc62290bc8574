"""The FP6 GEMM whose last partial round of 256 x 256 tiles runs as smaller workgroups: the
sums are exact in any order and the epilogue is shared, so its outputs are compared with the
plain 256 x 256 grid bit for bit (that grid is checked against the CPU oracle)."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(nat, args, M, N, K, dtype, res, gate):
    out = torch.full((M, N), float("nan"), dtype=dtype, device=args[0].device)
    nat.check(nat.load().convrot_w4a4_gemm_fp6_compact(
        *[nat.ptr(t) for t in args], M, N, K, nat.ptr(res), nat.ptr(gate), N if gate is not None else 0,
        (M + 1) // 2, nat.ptr(out), nat.dtype_code(dtype), nat.stream_of(out.device)))
    torch.cuda.synchronize()
    return out


# 270 tiles of 256 x 256, 14 past the first round: whole parts; column parts and row parts that are
# ragged or outside the output (116 columns, 48 rows in the last tiles); 512 + 8 tiles; one tile over.
@pytest.mark.parametrize("M,K,N", [(4608, 128, 3840), (4500, 640, 3700), (4400, 384, 3802), (10240, 128, 3328),
                                   (65700, 128, 203)])
@pytest.mark.parametrize("split", [None, "2", "4"])
def test_split_last_round_equals_plain_tiles(dev, tuning, split, M, K, N):
    from convrot_mlx_amd import _native as nat

    lib = nat.load()
    torch.manual_seed(M + K + N)
    x = torch.randn(M, K, device=dev).bfloat16()
    a6 = torch.zeros(int(lib.convrot_fp6_bytes(M, K)), dtype=torch.uint8, device=dev)
    xs = torch.empty(M, dtype=torch.float32, device=dev)
    nat.check(lib.convrot_prepare(nat.ptr(x), nat.dtype_code(x.dtype), M, K, 64, nat.PREP_FP6, nat.ptr(a6), nat.ptr(xs),
                                  nat.stream_of(dev)))
    nb = (N + 15) // 16
    w6 = torch.randint(0, 256, (K // 128 * nb * 1024,), dtype=torch.uint8, device=dev)
    ws = torch.rand(N, device=dev) + 0.1
    args = (a6, xs, w6, ws, torch.randn(N, device=dev))
    for dtype, gated in ((torch.bfloat16, False), (torch.float16, False), (torch.float32, False), (torch.bfloat16, True)):
        res = torch.randn(M, N, device=dev).to(dtype) if gated else None
        gate = torch.randn(2, N, device=dev).to(dtype) if gated else None
        tuning.set("fp6_tile", "256x256")
        want = _run(nat, args, M, N, K, dtype, res, gate)
        tuning.set("fp6_tile", None)
        tuning.set("fp6_split", split)
        got = _run(nat, args, M, N, K, dtype, res, gate)
        tuning.set("fp6_split", None)
        assert not torch.isnan(want).any()
        assert torch.equal(got, want), f"split {split}, {M}x{K}->{N} {dtype} gated={gated}"
