"""GPU: the training step's kernels at the edges of their tiles."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_surrogate import bf16_bits, bf16_value, run_gemm

pytestmark = pytest.mark.gpu


def gemm_bound(A, B, terms):
    """Largest error of an FP32 accumulation of exact products in any order: each of the `terms`
    roundings is at most 2^-24 (2^-23 allows for the matrix core's own rounding) of a partial sum,
    which the sum of magnitudes bounds."""
    return terms * 2.0 ** -23 * (np.abs(A) @ np.abs(B))


@pytest.mark.parametrize("M,N,K,splits", [
    (2, 128, 64, 2),          # one column pair, chunks of one 32-row step
    (224, 256, 96, 3),        # the first layer's 224 features: a ragged second tile
    (130, 128, 1344, 2),      # two columns past a tile, chunks of an odd number of steps
    (256, 256, 3072, 3),      # full tiles and chunks
    (256, 384, 8192, 8),      # three column tiles, one chunk to each XCD
])
def test_weight_gradient_gemm(M, N, K, splits):
    """dW = X^T dZ (A stored [K][M], B stored [K][N]) in split-K chunks, against numpy in FP64."""
    rng = np.random.default_rng(M + 3 * N + 5 * K)
    A, B = rng.normal(size=(K, M)).astype(np.float32), rng.normal(size=(K, N)).astype(np.float32)
    A16, B16 = bf16_bits(A), bf16_bits(B)
    a, b = bf16_value(A16).astype(np.float64).T, bf16_value(B16).astype(np.float64)
    print(f"[case] dW M={M} N={N} K={K} splits={splits}", flush=True)
    got, _ = run_gemm(A16, B16, M, N, K, 1, 0, splits)
    assert (np.abs(got - a @ b) <= gemm_bound(a, b, K + splits)).all()
