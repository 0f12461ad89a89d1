"""The quantizer's tiling (8 blocks of 4 rows per wave, 16-byte loads) and its
reciprocal path at their edges, byte for byte against the oracle."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,N,K,ldw", [(1, 32, 1, 32, 32), (3, 31, 4, 32, 33), (16, 256, 17, 288, 256),
                                          (17, 254, 17, 256, 255), (33, 1025, 40, 1088, 1031), (5, 2016, 5, 2048, 2019),
                                          (1000, 63, 1001, 64, 65), (130, 160, 133, 160, 161), (70, 320, 70, 320, 320),
                                          (70, 323, 71, 352, 323)])
def test_quantize_tile_edges(orc, dev, n, k, N, K, ldw):
    """Row and column remainders, waves that end one row and begin the next, row
    strides that are no multiple of 4, and
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


def test_quantize_row_of_2e31_columns(dev):
    """A row of 2^31 - 32 columns (1.3 GB of blocks): the column tiles are counted
    past 32 bits. One block of values, zero blocks with scale 1 after it."""
    import alveare_amd as aa

    print("\n[quantize] one row of 2^31 - 32 columns", flush=True)
    K = 2 ** 31 - 32
    src = torch.arange(-16.0, 16.0, device=dev).view(1, 32)
    got = aa.quantize_q4(src, 1, K).view(-1, 20)
    want = aa.quantize_q4(src, 1, 64).view(-1, 20)
    assert torch.equal(got[:2], want)
    for c in got[1:].split(1 << 24):
        assert torch.equal(c, want[1:].expand(c.shape[0], 20))
