"""GPU: the training step's kernels at the edges of their tiles."""
from __future__ import annotations

import numpy as np
import pytest

import linon_amd as L

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


def mix64(z):
    with np.errstate(over="ignore"):
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


GOLDEN = np.uint64(0x9E3779B97F4A7C15)


def training_set(seed, n, radius, inset):
    """The training set's entry states: a function of the seed (SplitMix64 stream)."""
    with np.errstate(over="ignore"):
        i = np.arange(6 * n, dtype=np.uint64)
        u = (mix64(np.uint64(seed) + GOLDEN * (i + np.uint64(1))) >> np.uint64(40)).astype(np.float64) * 2.0 ** -24
    u = u.reshape(n, 6)

    def direction(a, b):
        z, ph = 2.0 * u[:, a] - 1.0, 2.0 * np.pi * u[:, b]
        s = np.sqrt(np.maximum(0.0, 1.0 - z * z))
        return np.stack([s * np.cos(ph), s * np.sin(ph), z], 1)
    p, q = direction(0, 1), direction(2, 3)
    q[(p * q).sum(1) > 0] *= -1.0
    return np.concatenate([p * (radius - inset * u[:, 4:5]), q], 1).astype(np.float32)


def weights_of(blob):
    shapes = [s for k in (224, 256, 256, 256) for s in ((k, 256), (256,))] + [(256, 7), (7,)]
    flat = np.frombuffer(blob, np.float32, offset=len(blob) - 4 * sum(int(np.prod(s)) for s in shapes))
    cuts = np.cumsum([int(np.prod(s)) for s in shapes])[:-1]
    return [a.reshape(s).astype(np.float64) for a, s in zip(np.split(flat, cuts), shapes)]


def reference_gradients(w, x, target, conf_weight=0.1):
    """Loss gradients of the Fourier-feature MLP in FP64 (labels of the confidence all 0)."""
    freqs = np.pi / 2 * 32.0 ** (np.arange(16) / 15.0)
    a = freqs[None, :, None] * x[:, None, :]
    acts = [np.pad(np.concatenate([x, np.stack([np.sin(a), np.cos(a)], -1).reshape(len(x), -1)], 1), ((0, 0), (0, 26)))]
    zs = []
    for l in range(4):
        zs.append(acts[-1] @ w[2 * l] + w[2 * l + 1])
        acts.append(zs[-1] / (1.0 + np.exp(-zs[-1])))
    out = acts[4] @ w[8] + w[9]
    n = len(x)
    d = np.zeros_like(out)
    d[:, :6] = 2.0 * (out[:, :6] - target) / (6.0 * n)
    d[:, 6] = conf_weight / (1.0 + np.exp(-out[:, 6])) / n
    grads = [None] * 8 + [acts[4].T @ d, d.sum(0)]
    back = d @ w[8].T
    for l in (3, 2, 1, 0):
        s = 1.0 / (1.0 + np.exp(-zs[l]))
        dz = back * s * (1.0 + zs[l] * (1.0 - s))
        grads[2 * l], grads[2 * l + 1] = acts[l].T @ dz, dz.sum(0)
        back = dz @ w[2 * l].T
    return grads


@pytest.mark.parametrize("batch", [256, 320, 1088])  # whole row tiles; half a tile; a second chunk of 64 rows
def test_first_training_step(batch):
    """One step (gather, forward, loss, backward, gradients, Adam) from the initial weights.  Adam's
    first step moves every weight by -lr g / (|g| + 1e-8).  g is the FP64 gradient up to the BF16
    roundings of features, weights, activations and dZ (a dozen, 2^-9 each: about 1% of an array's
    RMS), so wherever |g| exceeds a tenth of the RMS the move has to be -lr sign(g)."""
    kw = dict(train_rays=2048, batch=batch, lr=1e-3, h=0.01, max_steps=1000, tolerance=1e-4, seed=7)
    print(f"[case] first training step, batch {batch}", flush=True)
    with L.MainView(16, 16) as view:
        view.train_surrogate(L.SurrogateConfig.make("swirl", steps=0, **kw))
        w0 = weights_of(view.save_surrogate())
        view.train_surrogate(L.SurrogateConfig.make("swirl", steps=1, **kw))
        w1 = weights_of(view.save_surrogate())
    states = training_set(7, 2048, 2.0, 0.01)
    ig = L.Integrator.make(h_initial=0.01, t_max=1e30, adaptive=False, max_steps=1000, mode=L.MODE_ESCAPE,
                           escape_radius=2.0, samples_per_ray=0, sample_steps=0, need_mapping=True, clip_exit=True)
    exits, _ = L.flowmap("swirl", ig, states)
    with np.errstate(over="ignore"):  # the mini-batch: hashed rows of the 1024 that are not held out
        i = np.arange(batch, dtype=np.uint64)
        rows = (mix64(np.uint64(7 ^ 0x5DEECE66D) + GOLDEN * (i + np.uint64(1))) % np.uint64(1024)).astype(np.int64)
    scale = np.array([0.5, 0.5, 0.5, 1.0, 1.0, 1.0])
    grads = reference_gradients(w0, states[rows].astype(np.float64) * scale, exits[rows].astype(np.float64) * scale)
    for k, (a, b, g) in enumerate(zip(w0, w1, grads)):
        clear = np.abs(g) > 0.1 * np.sqrt((g * g).mean())
        move = (b - a)[clear]
        # FP32 weights: a move carries the rounding of the weight itself
        assert clear.any() and (np.abs(move + 1e-3 * np.sign(g[clear])) <= 1e-5 + 2.0 ** -23 * np.abs(a[clear])).all(), k
        # the padding rows of the first layer have no gradient and stay
        if k == 0:
            assert np.array_equal(b[198:], a[198:])


# the sums' unrolled pieces: 8 rows and one more; 16 rows for some of the 256 sums and not for others;
# 18 chunks, so that the update adds 16 partials and two single ones
@pytest.mark.parametrize("batch", [2112, 4160, 17472])
def test_first_step_of_a_large_batch(batch):
    test_first_training_step(batch)


@pytest.mark.parametrize("batch", [0, 255, 288, 1056])
def test_batches_of_other_than_whole_chunks_are_refused(batch):
    """The gradient tiles read whole steps of 32 rows of chunks that end with the batch."""
    with L.MainView(16, 16) as view:
        with pytest.raises(L.LinonError, match="bad configuration"):
            view.train_surrogate(L.SurrogateConfig.make("swirl", steps=1, train_rays=2048, batch=batch, lr=1e-3,
                                                        h=0.01, max_steps=1000, tolerance=1e-4, seed=7))
