"""GPU parity: the preparation of 16-bit activations on packed registers, where it can go wrong."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import from_dev, to_dev

pytestmark = pytest.mark.gpu


def _unblocked(blocks, M, K):
    """Row-major codes of PREP_INT8_BLOCKED blocks: [kb, mb, s, q, r, b] -> row 16 mb + r, feature 128 kb + 32 q + 16 s + b."""
    kb, mb, _ = blocks.shape
    return blocks.reshape(kb, mb, 2, 4, 16, 16).transpose(1, 4, 0, 3, 2, 5).reshape(mb * 16, kb * 128)[:M, :K]


def _check(orc, dev, x16, dtype, G):
    """Codes and scales of the int8, packed, blocked and FP6 outputs against the oracle's."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    M, K = x16.shape
    codes, scales = orc.prepare_codes(x16, dtype, G)
    x = to_dev(x16, dtype, dev)
    got, s = core._prepare(x, G, nat.PREP_INT8)
    assert np.array_equal(from_dev(got), codes) and np.array_equal(from_dev(s), scales)
    got, s = core._prepare(x, G, nat.PREP_PACKED)
    assert np.array_equal(from_dev(got), orc.pack_signed_int4(codes)) and np.array_equal(from_dev(s), scales)
    got, s = core._prepare(x, G, nat.PREP_INT8_BLOCKED)
    assert np.array_equal(_unblocked(from_dev(got), M, K), codes) and np.array_equal(from_dev(s), scales)
    if K % 128 == 0:
        got, s = core._prepare(x, G, nat.PREP_FP6)
        assert np.array_equal(orc.fp6_to_codes(from_dev(got), M, K), codes) and np.array_equal(from_dev(s), scales)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("G", [4, 16, 64, 256, 1024])
@pytest.mark.parametrize("ni", [1, 3, 4])
def test_magnitudes(orc, dev, tuning, dtype, G, ni):
    """Every group size and iteration count on rows of every magnitude: the format's smallest denormals,
    values 2^20 apart in one group (sums that round), the largest that stay finite, zeros of both signs."""
    tuning.set("prep_ni", ni)
    rng = np.random.default_rng(G + ni)
    K = 5120
    top = 2.0 ** (90 if dtype == "bfloat16" else 4)
    rows = [rng.normal(size=K) * s for s in (1.0, top, 2.0 ** -24, 2.0 ** -20, 2.0 ** -14)]
    rows.append(rng.normal(size=K) * 2.0 ** rng.integers(-20, 3, size=K))
    rows.append(np.where(rng.random(K) < 0.5, -0.0, 0.0))
    rows.append(rng.integers(-3, 4, size=K) * 2.0 ** -24)
    if dtype == "bfloat16":
        rows += [rng.normal(size=K) * 2.0 ** -130, rng.integers(-2, 3, size=K) * 2.0 ** -133]
    with np.errstate(over="ignore"):
        x16 = orc.from_f32(np.array(rows, dtype=np.float32), dtype)
    _check(orc, dev, x16, dtype, G)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("mode", ["int8", "fp6", "blocked", "packed"])
def test_nonfinite_rows(dev, dtype, mode):
    """Infinities, NaN and sums that overflow: the bits of the float32 kernel's arithmetic (a float16 or
    bfloat16 row prepared without rotation after an eager rotation in the dtype), rows beside them untouched."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    kind = {"int8": nat.PREP_INT8, "fp6": nat.PREP_FP6, "blocked": nat.PREP_INT8_BLOCKED, "packed": nat.PREP_PACKED}[mode]
    dt = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    M, K, G = 6, 4096, 256
    x = torch.randn(M, K, device=dev)
    big = 3e38 if dtype == "bfloat16" else 6e4
    x[1, 70], x[2, 3000], x[2, 3001], x[3, :] = float("inf"), float("-inf"), float("inf"), big
    x[4, 5], x[4, 2000] = float("nan"), 9.0
    x = x.to(dt)
    got, scales = core._prepare(x, G, kind)

    def rotate(v):  # the eager butterfly, every sum rounded to the dtype
        stride = 1
        while stride < G:
            a, b, c, d = v.reshape(M, K // (4 * stride), 4, stride).unbind(2)
            v = torch.stack([a + b + c - d, a + b - c + d, a - b + c + d, -a + b + c + d], 2).reshape(M, K)
            stride *= 4
        return (v.float() / 16).to(dt)

    want, want_scales = core._prepare(rotate(x), 1, kind | nat.PREP_NO_ROTATE)
    assert torch.equal(scales.nan_to_num(1.5), want_scales.nan_to_num(1.5))
    if mode == "fp6":  # [kb, 1, 16 bytes of a (q, row) slot]; a NaN's field has the NaN's sign, which torch's may not
        rows = lambda t: t[:, 0, :1024].reshape(K // 128, 4, 16, 16)[:, :, :M]  # noqa: E731
        nan = torch.isnan(rotate(x).float() / scales[:, None])
        clean = ~nan.reshape(M, K // 128, 4, 32).any(-1).permute(1, 2, 0)
        assert torch.equal(rows(got)[clean], rows(want)[clean])
    elif mode == "blocked":
        rows = lambda t: t.reshape(K // 128, 2, 4, 16, 16)[:, :, :, :M]  # noqa: E731
        assert torch.equal(rows(got), rows(want))
    else:
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
def test_gelu_every_value(orc, dev, dtype):
    """Every 16-bit input with finite sums through the GELU producer: the oracle's codes (the reciprocal and the
    exponent arithmetic at every significand and range), and a head in front."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    bits = np.arange(65536, dtype=np.uint16)
    # below an eighth of the largest value, so that the sums of a group stay finite
    bits = bits[np.abs(orc.to_f32(bits, dtype)) < (2.0 ** 124 if dtype == "bfloat16" else 2.0 ** 12)]
    order = np.argsort(np.abs(orc.to_f32(bits, dtype)), kind="stable")  # rows of like magnitudes: codes of all of them
    bits = bits[order][: bits.size // 256 * 256].reshape(-1, 256)
    head = np.ascontiguousarray(bits[:, :64])
    x16 = orc.gelu_producer_rows(None, bits, dtype)
    codes, scales = orc.prepare_codes(x16, dtype, 4)
    got, s = core._prepare_gelu(to_dev(bits, dtype, dev), None, 4, nat.PREP_INT8)
    assert np.array_equal(from_dev(got), codes) and np.array_equal(from_dev(s), scales)
    x16 = orc.gelu_producer_rows(head, bits, dtype)
    codes, scales = orc.prepare_codes(x16, dtype, 64)
    got, s = core._prepare_gelu(to_dev(bits, dtype, dev), to_dev(head, dtype, dev), 64, nat.PREP_PACKED)
    assert np.array_equal(from_dev(got), orc.pack_signed_int4(codes)) and np.array_equal(from_dev(s), scales)


@pytest.mark.parametrize("dtype,G,M,K,mode,cut", [("bfloat16", 64, 2080, 13312, "fp6", 1040),
                                                  ("bfloat16", 64, 2080, 8192, "fp6", 1040),
                                                  ("bfloat16", 16, 1600, 8192, "fp6", 800),
                                                  ("float16", 16, 2080, 16384, "fp6", 1040),
                                                  ("float16", 64, 2000, 12288, "rotate", 1000)])
def test_routes_agree(dev, tuning, dtype, G, M, K, mode, cut):
    """The automatic kernel and split of all the rows, and those of a part of them with every number of
    iterations: other routes, the same bytes."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    dt = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    kind = {"fp6": nat.PREP_FP6, "rotate": nat.PREP_ROTATE}[mode]
    plan = lambda m: nat.prepare_plan(m, K, nat.dtype_code(dt), G, kind)  # noqa: E731
    x = (torch.randn(M, K, device=dev) * 3).to(dt)
    route = plan(M)
    whole, s = core._prepare(x, G, kind)
    others = set()
    for ni in (None, 1, 3, 4):
        tuning.set("prep_ni", ni)
        others.add(plan(cut))
        for i in range(0, M, cut):
            part, sp = core._prepare(x[i : i + cut], G, kind)
            if mode == "rotate":
                assert torch.equal(whole[i : i + cut].view(torch.int16), part.view(torch.int16))
            else:
                assert torch.equal(whole[:, i // 16 : (i + cut) // 16], part) and torch.equal(s[i : i + cut], sp)
    tuning.set("prep_ni", None)
    assert len(others - {route}) >= 2


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("producer", ["plain", "modulated", "gelu", "gelu head"])
@pytest.mark.parametrize("G,ni", [(4, 1), (16, 4), (64, None), (64, 3), (256, 1), (256, 4), (1024, 3)])
def test_nonfinite_producers(orc, dev, tuning, dtype, producer, G, ni):
    """Rows with infinities, NaN and overflows behind every producer, in every output: the oracle's produced
    rows, rotated eagerly in the dtype and quantized by the kernel without a rotation; clean rows beside them."""
    from convrot_mlx_amd import _native as nat
    from convrot_mlx_amd import core

    tuning.set("prep_ni", ni)
    dt = {"bfloat16": torch.bfloat16, "float16": torch.float16}[dtype]
    M, K = 7, 4096
    rng = np.random.default_rng(G + (ni or 0))
    big = np.float32(3e38 if dtype == "bfloat16" else 6e4)
    x = rng.normal(size=(M, K)).astype(np.float32)
    wild = rng.normal(size=(M, K)).astype(np.float32)  # the non-finite values go in here
    wild[1, 70], wild[2, 3000], wild[2, 3001] = np.inf, np.inf, np.inf
    wild[3, :], wild[4, 5], wild[4, 2000], wild[5, 1024:2048] = big, np.nan, 9.0, -big
    bits = lambda v: orc.from_f32(v.astype(np.float32), dtype)  # noqa: E731
    if producer == "plain":
        wild[2, 3001] = -np.inf
        rows16 = bits(wild)
        prep = lambda kind: core._prepare(to_dev(rows16, dtype, dev), G, kind)  # noqa: E731
    elif producer == "modulated":  # a vector a row: products and sums overflow, (1 + inf) * 0 is NaN
        x16, sh16, sc16 = bits(x), bits(rng.normal(size=(M, K))), bits(wild)
        rows16 = orc.modulate(x16, dtype, sh16, sc16, 1)
        xt, sht, sct = (to_dev(v, dtype, dev) for v in (x16, sh16, sc16))
        prep = lambda kind: core._prepare_modulated(xt, sht, sct, G, kind, 1e-6)  # noqa: E731
    else:
        kh = 1024 if producer == "gelu head" else 0
        w16 = bits(wild)
        head, x16 = (np.ascontiguousarray(w16[:, :kh]), np.ascontiguousarray(w16[:, kh:])) if kh else (None, w16)
        rows16 = orc.gelu_producer_rows(head, x16, dtype)
        ht, xt = None if head is None else to_dev(head, dtype, dev), to_dev(x16, dtype, dev)
        prep = lambda kind: core._prepare_gelu(xt, ht, G, kind)  # noqa: E731
    v, stride = to_dev(rows16, dtype, dev), 1
    assert not torch.isfinite(v).all(1)[[1, 4]].any() and torch.isfinite(v).all(1)[[0, 6]].all()
    while stride < G:
        a, b, c, d = v.reshape(M, K // (4 * stride), 4, stride).unbind(2)
        v = torch.stack([a + b + c - d, a + b - c + d, a - b + c + d, -a + b + c + d], 2).reshape(M, K)
        stride *= 4
    rotated = (v.float() / G ** 0.5).to(dt)
    got = prep(nat.PREP_ROTATE)[0]
    assert torch.equal(torch.isnan(got), torch.isnan(rotated))
    assert torch.equal(got.nan_to_num(0.0, 7e4, -7e4), rotated.nan_to_num(0.0, 7e4, -7e4))
    for kind in (nat.PREP_INT8, nat.PREP_PACKED, nat.PREP_INT8_BLOCKED, nat.PREP_FP6):
        got, scales = prep(kind)
        want, want_scales = core._prepare(rotated, 1, kind | nat.PREP_NO_ROTATE)
        assert torch.equal(scales.nan_to_num(1.5), want_scales.nan_to_num(1.5))
        if kind == nat.PREP_INT8_BLOCKED:
            assert np.array_equal(_unblocked(from_dev(got), M, K), _unblocked(from_dev(want), M, K))
        elif kind != nat.PREP_FP6:
            assert torch.equal(got, want)
        else:  # both parts of a 32-feature slot; a NaN's field has the NaN's sign, which torch's may not
            nan = torch.isnan(rotated.float() / scales[:, None])
            clean = ~nan.reshape(M, K // 128, 4, 32).any(-1).permute(1, 2, 0)
            for lo, hi, width in ((0, 1024, 16), (1024, 1536, 8)):
                part = lambda t: t[:, 0, lo:hi].reshape(K // 128, 4, 16, width)[:, :, :M]  # noqa: B023, E731
                assert torch.equal(part(got)[clean], part(want)[clean])
            assert clean[:, :, [0, 6]].all()
