"""GPU parity: the 16-byte NK <-> CDNA4 repack at the edges of its blocks, and where the byte-wise one stays."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _util import from_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 16, 17, 95])
@pytest.mark.parametrize("K", [32, 128, 160, 512, 544, 672])
def test_repack_edges(orc, dev, N, K):
    """Rows that end inside a block of 16, features that end on any 32 of a 128-feature block and on
    any block of a wave's four; every nibble value.  Bytes are exact, padding is zero."""
    import convrot_mlx_amd as api

    rng = np.random.default_rng(1000 * N + K)
    v = rng.integers(-8, 8, size=(N, K), dtype=np.int8)
    nk = orc.pack_signed_int4(v)
    c4 = api.repack_nk_weight_for_cdna4(torch.from_numpy(nk).to(dev))
    assert np.array_equal(from_dev(c4), orc.codes_to_cdna4(v))
    assert np.array_equal(from_dev(api.repack_cdna4_weight_to_nk(c4, N, K)), nk)


@pytest.mark.parametrize("N,K,offset", [(33, 50, 0), (33, 16, 0), (34, 256, 4), (18, 64, 1)])
def test_repack_bytewise(orc, dev, N, K, offset):
    """Rows that are not whole 16-byte pieces, and buffers that do not start on 16 bytes."""
    import convrot_mlx_amd as api

    rng = np.random.default_rng(N * K + offset)
    v = rng.integers(-8, 8, size=(N, K), dtype=np.int8)
    nk = orc.pack_signed_int4(v)
    buf = torch.zeros(offset + nk.size, dtype=torch.uint8, device=dev)
    view = buf[offset:].view(nk.shape)
    view.copy_(torch.from_numpy(nk))
    c4 = api.repack_nk_weight_for_cdna4(view)
    assert np.array_equal(from_dev(c4), orc.codes_to_cdna4(v))
    buf4 = torch.zeros(offset + c4.numel(), dtype=torch.uint8, device=dev)
    view4 = buf4[offset:].view(c4.shape)
    view4.copy_(c4)
    assert np.array_equal(from_dev(api.repack_cdna4_weight_to_nk(view4, N, K)), nk)
