"""The support product's tiles (-m gpu): the order of the tiles over the XCDs,
K of one to several K tiles, ragged edges.  Weights of small whole numbers and
0/1 spikes: every sum is exact, so the result equals the integer product."""

import numpy as np
import pytest

from test_gpu_recall import _bf16_bits, _gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,N,K", [
    (1, 1, 64),          # one small tile, one K tile
    (64, 64, 128),       # exactly one
    (65, 63, 192),       # a row past it, a column short
    (705, 513, 64),      # 12 x 9 small tiles: a group of four row tiles, 108 over 8 XCDs
    (255, 4097, 320),    # 4 x 65 small tiles
    (4097, 1793, 64),    # 17 x 8 large tiles: a group of one row tile, one K tile
    (2816, 2816, 128),   # 11 x 11: small
    (2817, 2816, 192),   # 12 x 11: large, a row past a tile
    (257, 16640, 320),   # 2 x 65 large tiles, 130 over 8 XCDs
])
def test_tiles(B, N, K):
    rng = np.random.Generator(np.random.Philox(B + N + K))
    S = (rng.random((B, K)) < 0.3).astype(np.float32)
    W = rng.integers(-8, 9, size=(N, K)).astype(np.float32)
    E = rng.integers(-64, 65, size=(B, N)).astype(np.float32)
    got = _gemm(_bf16_bits(S), _bf16_bits(W), E, 0.5)
    assert np.array_equal(got, (np.float32(0.5) * E + S @ W.T).astype(np.float32))
