"""The quantizer's tiling (4 rows x 256 columns per wave, 16-byte loads) and its
reciprocal path at their edges, byte for byte against the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,N,K,ldw", [(1, 32, 1, 32, 32), (3, 31, 4, 32, 33), (16, 256, 17, 288, 256),
                                          (17, 254, 17, 256, 255), (33, 1025, 40, 1088, 1031), (5, 2016, 5, 2048, 2019)])
def test_quantize_tile_edges(orc, dev, n, k, N, K, ldw):
    """Row and column remainders, row strides that are no multiple of 4, and
    quotients at and within a few ulps of every half integer, where the
    reciprocal cannot settle the code and the division must."""
    import alveare_amd as aa

    print(f"\n[quantize] {n}x{k} -> {N}x{K}, rows {ldw} apart", flush=True)
    rng = np.random.default_rng(n * k)
    w = rng.normal(0.0, 0.02, size=(n, ldw)).astype(np.float32)
    # Every other row: the block maximum m, then (h + 1/2) m / 7 a few ulps up and down.
    m = rng.uniform(0.01, 3.0, size=(n, 1)).astype(np.float32)
    half = (rng.integers(-7, 7, size=(n, ldw)) + np.float32(0.5)).astype(np.float32) * (m / np.float32(7.0))
    half = (half.view(np.int32) + rng.integers(-3, 4, size=half.shape).astype(np.int32)).view(np.float32)
    half[:, ::32] = m
    w[::2] = half[::2]
    w[n // 2] *= np.float32(1e-33)  # scales outside the reciprocal's range
    src = torch.from_numpy(w).to(dev)[:, :k]
    got = aa.quantize_q4(src, N, K).cpu().numpy()
    pad = np.zeros((N, K), np.float32)
    pad[:n, :k] = w[:, :k]
    assert np.array_equal(got, orc.quantize_q4_0(pad))
