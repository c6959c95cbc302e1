"""The fused network against the launches it stands for, at the edges of its 128-row tiles."""
from __future__ import annotations

import numpy as np
import pytest

import linon_amd as L
from linon_amd import configs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def view():
    view = L.MainView(64, 64)
    view.load_surrogate(configs.saved_surrogate("hot_air"))
    return view


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 255, 257])
def test_fused_inference_at_tile_edges(view, n):
    """The same bits as a kernel a layer; the first states twice as far out and a zero direction, so
    that activations reach both ends of the SiLU."""
    rng = np.random.default_rng(n)
    states = rng.normal(size=(n, 6)).astype(np.float32)
    states[: n // 4, :3] *= 1e3
    states[0, 3:] = 0.0
    print(f"[case] {n} states", flush=True)
    fused, plain = view.surrogate_infer(states, fused=True), view.surrogate_infer(states, fused=False)
    assert np.isfinite(plain).all()
    np.testing.assert_array_equal(fused, plain)
