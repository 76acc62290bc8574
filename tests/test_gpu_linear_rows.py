"""GPU parity: the one-launch linear of a few rows against the oracle (W4A4) and the two launches (W4A16)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import from_dev, outlier_input, to_dev

pytestmark = pytest.mark.gpu

DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def _layer(orc, dev, K, N, G, backend, seed):
    import convrot_mlx_amd as api

    rng = np.random.default_rng(seed)
    w = orc.from_f32((rng.normal(size=(N, K)) * 0.02).astype(np.float32), "bfloat16")
    layer = api.ConvRotLinear(K, N, group_size=G, backend=backend, device=dev)
    qw, ws = api.quantize_convrot_weight(to_dev(w, "bfloat16", dev), G)
    bias = rng.normal(size=N).astype(np.float32)
    layer.load_nk_weight(qw, ws, torch.from_numpy(bias).to(dev))
    return layer, orc.unpack_signed_int4(from_dev(qw)), from_dev(ws), bias


def _two_launches(api, layer, x, **residual):
    """The layer's product through its preparation and GEMM entry points."""
    if layer.a4:
        a, xs = api.hip_fused_prepare_convrot_activation_i8(x, layer.group_size)
        return api.hip_w4a4_int8_matmul(a, layer.qweight, xs, layer.scales, layer.bias, output_dtype=x.dtype,
                                        out_features=layer.out_features, **residual)
    a = api.hip_fused_rotate_convrot_activation(x, layer.group_size)
    return api.hip_w4a16_matmul(a, layer.qweight, layer.scales, layer.bias, output_dtype=x.dtype,
                                out_features=layer.out_features, **residual)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16", "float32"])
@pytest.mark.parametrize("M,K,N,G", [(1, 64, 1, 64), (1, 192, 33, 64), (2, 2880, 50, 64), (4, 1024, 272, 256),
                                     (3, 1280, 4100, 256), (1, 8192, 48, 256), (1, 3072, 8200, 64)])
def test_w4a4_rows(orc, dev, dtype, M, K, N, G):
    """Codes, dots and outputs are the oracle's bits: a row shorter than a wave's block, K ending
    inside a 128-feature block and inside a wave's 1024, N off the vector stores and the tile
    groups, several batches of k-blocks, and (8200) a third tile a workgroup."""
    layer, w_codes, ws, bias = _layer(orc, dev, K, N, G, "hip-w4a4", M * K + N)
    from convrot_mlx_amd import core

    x = outlier_input(K + N, (M, K), dtype, orc)
    xt = to_dev(x, dtype, dev)
    got = core._linear_rows(xt, G, True, layer.qweight, layer.scales, layer.bias, N, None)
    a_codes, xs = orc.prepare_codes(x, dtype, G)
    want = orc.w4a4_matmul_codes(a_codes, w_codes, xs, ws, bias, dtype)
    assert np.array_equal(from_dev(got).view(np.uint8), np.ascontiguousarray(want).view(np.uint8))


@pytest.mark.parametrize("cfg", [1, 2, 3, 5, 16])
@pytest.mark.parametrize("backend", ["hip-w4a4", "hip-w4a16"])
def test_rows_every_split(orc, dev, tuning, cfg, backend):
    """Every split against the two launches, with more tile groups than workgroups (N = 20832: 1302
    tiles), a ragged last k-block and batch, a gated residual, and poisoned bytes behind the rows."""
    import convrot_mlx_amd as api
    from convrot_mlx_amd import core

    K, N, G, M = 3904, 20832, 64, 2
    layer, *_ = _layer(orc, dev, K, N, G, backend, cfg)
    buf = torch.full((M * K + 4096,), float("nan"), dtype=torch.bfloat16, device=dev)
    x = buf[: M * K].view(M, K)
    x.copy_(torch.randn(M, K, device=dev))
    residual = torch.randn(M, N, device=dev).bfloat16()
    gate = torch.randn(1, N, device=dev).bfloat16()
    want = _two_launches(api, layer, x, residual=residual, gate=gate)
    tuning.set("linear_rows_cfg", cfg)
    gr = core._gated_residual(residual, gate, (M, N), torch.bfloat16)
    got = core._linear_rows(x, G, layer.a4, layer.qweight, layer.scales, layer.bias, N, gr)
    if layer.a4:
        assert torch.equal(got, want)
    else:
        # float32 sums of at most 31 x 128 products in another order: a few results cross a rounding of
        # the linear, its product with the gate and the sum, at most one step of each
        step = 2.0 ** -8
        lin = _two_launches(api, layer, x).float()
        bound = 2 * step * ((lin * gate.float()).abs() * 2 + want.float().abs())
        assert ((got.float() - want.float()).abs() <= bound).all()
        assert (got != want).float().mean() < 1e-3


@pytest.mark.parametrize("backend,dtype", [("hip-w4a4", "bfloat16"), ("hip-w4a4", "float32"),
                                           ("hip-w4a16", "bfloat16"), ("hip-w4a16", "float16")])
def test_layer_route(orc, dev, backend, dtype):
    """ConvRotLinear on either side of the rule: shapes of 0 to 9 rows, non-contiguous x, the in-place
    residual (x itself the residual), equal to the two launches."""
    import convrot_mlx_amd as api

    K = N = 1024
    layer, *_ = _layer(orc, dev, K, N, 256, backend, 7)
    dt = DTYPES[dtype]
    for lead in [(0,), (1,), (1, 1), (2, 2), (5,), (9,)]:
        x = torch.randn(*lead, 2 * K, device=dev).to(dt)[..., :K]  # row stride 2 K
        got = layer(x)
        assert got.shape == (*lead, N) and got.dtype == dt
        x2d = x.reshape(-1, K)
        if x2d.shape[0] == 0:
            continue
        want = _two_launches(api, layer, x2d).reshape(got.shape)
        if layer.a4:
            assert torch.equal(got, want)
        else:  # one step of the output type where a float32 sum lies beside a rounding boundary
            ulp = 2.0 ** -7 if dtype == "bfloat16" else 2.0 ** -10
            assert ((got.float() - want.float()).abs() <= ulp * want.float().abs() + 1e-6).all()
        own = x.contiguous()
        plain = layer(own, residual=own.clone())
        res = own.clone()
        assert layer(res, residual=res, inplace=True) is res
        if layer.a4:
            assert torch.equal(res, plain)


def test_rows_nonfinite(orc, dev):
    """Rows with infinities and NaN: the same bits as the two launches, and other rows untouched."""
    import convrot_mlx_amd as api
    from convrot_mlx_amd import core

    K, N, G = 1024, 96, 64
    for backend in ("hip-w4a4", "hip-w4a16"):
        layer, *_ = _layer(orc, dev, K, N, G, backend, 3)
        x = torch.randn(4, K, device=dev).bfloat16()
        x[1, 5] = float("inf")
        x[2, 700] = float("nan")
        x[3] = 3e38
        want = _two_launches(api, layer, x)
        got = core._linear_rows(x, G, layer.a4, layer.qweight, layer.scales, layer.bias, N, None)
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got.nan_to_num(0.0)[0], want.nan_to_num(0.0)[0])
        if layer.a4:
            assert torch.equal(got.nan_to_num(0.0), want.nan_to_num(0.0))


@pytest.mark.parametrize("backend", ["hip-w4a4", "hip-w4a16"])
@pytest.mark.parametrize("M", [1, 3, 4, 8])
def test_inplace_bits(orc, dev, backend, M):
    """In place and out of place are the same bits: a residual of its own, x itself, and a residual that
    starts inside x or in which x starts; x is read before any of it is written."""
    K = N = 1024
    layer, *_ = _layer(orc, dev, K, N, 256, backend, M)
    gate = torch.randn(1, N, device=dev).bfloat16()
    for offset in (None, 0, 8, N // 2 + 8, -8, -(N // 2)):  # elements from x's start to the residual's
        for g in (None, gate):
            buf = torch.randn(2 * M * N + N, device=dev).bfloat16()
            x = buf[N // 2 :][: M * K].view(M, K)
            start = N // 2 + offset if offset is not None else N // 2 + M * K
            res = buf[start :][: M * N].view(M, N)
            want = layer(x.clone(), residual=res.clone(), gate=g)
            assert layer(x, residual=res, gate=g, inplace=True) is res
            assert torch.equal(res, want), (offset, g is None)


@pytest.mark.parametrize("backend", ["hip-w4a4", "hip-w4a16"])
def test_few_rows_make_the_workspace(orc, dev, backend):
    """A stream whose eager calls had one row has its workspace: a later capture of more rows runs the plan
    (and, W4A16, the bits) of an eager call of those rows."""
    from convrot_mlx_amd import core

    layer, *_ = _layer(orc, dev, 12288, 512, 256, backend, 5)
    x = torch.randn(32, 12288, device=dev).bfloat16()
    want = layer(x)
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    core._WORKSPACES.pop((stream.device.index, stream.cuda_stream), None)
    with torch.cuda.stream(stream):
        layer(x[:1])
    torch.cuda.synchronize()
    assert (stream.device.index, stream.cuda_stream) in core._WORKSPACES
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        got = layer(x)
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
