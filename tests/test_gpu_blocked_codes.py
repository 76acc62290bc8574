"""GPU parity: blocked int8 codes (CONVROT_PREP_INT8_BLOCKED) and the W4A4 kernel that reads them."""

from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SPLITS = [21, 22, 23, 24, 31, 32, 33, 43, 52]
DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def _rows(blocks: torch.Tensor, m: int, k: int) -> torch.Tensor:
    """Row-major codes of the blocks: [kb, mb, s, q, r, b] -> row 16 mb + r, feature 128 kb + 32 q + 16 s + b."""
    kb, mb, _ = blocks.shape
    return blocks.view(kb, mb, 2, 4, 16, 16).permute(1, 4, 0, 3, 2, 5).reshape(mb * 16, kb * 128)[:m, :k]


@pytest.mark.parametrize("dtype", list(DTYPES))
@pytest.mark.parametrize("M,K,G", [(5, 64, 64), (16, 1472, 64), (77, 3072, 256), (33, 1024, 1024), (7, 5120, 16)])
def test_blocked_prep(dev, dtype, M, K, G):
    """Every producer writes the codes and scales of the row-major mode, in blocks: ragged rows, K ending
    inside a block, every exchange layout."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    dt = DTYPES[dtype]
    x = (torch.randn(M, K, device=dev) * 3).to(dt)
    sh, sc = (torch.randn(1, K, device=dev).to(dt) for _ in range(2))
    head = torch.randn(M, K // 4 // 16 * 16, device=dev).to(dt)
    for prep in (lambda mode: core._prepare(x, G, mode), lambda mode: core._prepare_modulated(x, sh, sc, G, mode, 1e-6),
                 lambda mode: core._prepare_gelu(x[:, : K - head.shape[1]], head, G, mode)):
        codes, scales = prep(nat.PREP_INT8)
        blocks, scales_b = prep(nat.PREP_INT8_BLOCKED)
        assert tuple(blocks.shape) == (-(-K // 128), -(-M // 16), 2048)
        assert torch.equal(_rows(blocks, M, K), codes) and torch.equal(scales, scales_b)


@pytest.mark.parametrize("split", SPLITS)
@pytest.mark.parametrize("M,K,N", [(5, 64, 7), (33, 1472, 50), (81, 1024, 272), (129, 2688, 97), (255, 1152, 64)])
def test_every_split(orc, dev, tuning, split, M, K, N):
    """Every split against the oracle, with garbage in the blocks' padding rows and features: part tiles in
    rows and columns, fewer k-blocks than waves, N off the vector stores, -8 weights."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    rng = np.random.default_rng(split * 1000 + M)
    a = rng.integers(-8, 8, size=(M, K), dtype=np.int8)
    w = rng.integers(-8, 8, size=(N, K), dtype=np.int8)
    xs, ws = (rng.uniform(0.01, 0.2, size=n).astype(np.float32) for n in (M, N))
    bias = rng.normal(size=N).astype(np.float32)
    padded = rng.integers(-128, 128, size=(-(-M // 16) * 16, -(-K // 128) * 128), dtype=np.int8)
    padded[:M, :K] = a
    blocks = padded.reshape(-1, 16, padded.shape[1] // 128, 4, 2, 16).transpose(2, 0, 4, 3, 1, 5)
    act = torch.from_numpy(np.ascontiguousarray(blocks).reshape(blocks.shape[0], blocks.shape[1], 2048)).to(dev)
    wq = torch.from_numpy(orc.codes_to_cdna4(w)).to(dev)
    to = lambda v: torch.from_numpy(v).to(dev)  # noqa: E731
    tuning.set("w4a4_midm_cfg", split)
    for dtype, dt in DTYPES.items():
        got = core._w4a4(act, nat.ACT_INT8_BLOCKED, K, wq, to(xs), to(ws), to(bias), dt, N, None, M)
        want = orc.w4a4_matmul_codes(a, w, xs, ws, bias, dtype)
        assert np.array_equal(got.cpu().view(torch.uint8).numpy().reshape(-1),
                              np.ascontiguousarray(want).view(np.uint8).reshape(-1)), dtype


@pytest.mark.parametrize("M,K,N,G", [(5, 1024, 8208, 64), (16, 1024, 1024, 64), (100, 3072, 3000, 256), (255, 1472, 1000, 64)])
@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
def test_layer_route(dev, dtype, M, K, N, G):
    """ConvRotLinear on blocked codes, with and without a gated residual (in place too), equals its
    row-major products."""
    import convrot_mlx_amd as api
    from convrot_mlx_amd import core

    dt = DTYPES[dtype]
    layer = api.ConvRotLinear(K, N, group_size=G, backend="hip-w4a4", device=dev)
    layer.load_nk_weight(*api.quantize_convrot_weight((torch.randn(N, K, device=dev) * 0.02).bfloat16(), G),
                         torch.randn(N, device=dev))
    assert core._blocked_codes(M, N, K)
    x, res = torch.randn(M, K, device=dev).to(dt), torch.randn(M, N, device=dev).to(dt)
    gate = torch.randn(N, device=dev).to(dt)
    a, xs = api.hip_fused_prepare_convrot_activation_i8(x, G)
    for kw in ({}, {"residual": res}, {"residual": res, "gate": gate}):
        want = api.hip_w4a4_int8_matmul(a, layer.qweight, xs, layer.scales, layer.bias, output_dtype=dt,
                                        out_features=N, **kw)
        assert torch.equal(layer(x, **kw), want)
    own = res.clone()
    assert layer(x, residual=own, gate=gate, inplace=True) is own and torch.equal(own, want)
