"""The loop of fixed steps without a mesh against the general loop, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import linon_amd as L

pytestmark = pytest.mark.gpu


def states(n, radius, seed):
    rng = np.random.default_rng(seed)
    p, q = rng.normal(size=(2, n, 3))
    p *= radius / np.linalg.norm(p, axis=1, keepdims=True)
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    return np.concatenate([p, q], axis=1).astype(np.float32)


@pytest.mark.parametrize("weight", [1.0, 0.5])
@pytest.mark.parametrize("clip_exit", [0, 1])
@pytest.mark.parametrize("math", [L.MATH_IEEE, L.MATH_WGSL])
@pytest.mark.parametrize("field", ["identity", "swirl", "lens", "hot_air", "warp", "mirage_spherical_sigmoid"])
def test_fixed_steps_equal_the_general_loop(field, math, clip_exit, weight):
    """At h = 0.002 the adaptive rule never changes the step, so an adaptive integrator, which takes
    the general loop, makes the same steps.  Caps of 1 to 4 steps and a long one, from within the
    sphere, from just inside it, from on it and from outside; 65 rays, so that the second wave has
    one, two of them without a direction or a position."""
    for cap in (1, 2, 3, 4, 1501):
        ig = [L.Integrator.make(h_initial=0.002, t_max=1e30, adaptive=adaptive, max_steps=cap, mode=L.MODE_ESCAPE,
                                escape_radius=2.0, samples_per_ray=0, sample_steps=0, need_mapping=True,
                                clip_exit=bool(clip_exit)) for adaptive in (False, True)]
        for radius in (1.0, 1.998, 2.0, 2.3):
            s = states(65, radius, seed=cap)
            s[3, 3:] = 0.0
            s[5, :3] = 0.0
            print(f"[case] {field} math {math} clip {clip_exit} weight {weight} cap {cap} from {radius}", flush=True)
            got, steps = L.flowmap(field, ig[0], s, field_weight=weight, math=math)
            want, want_steps = L.flowmap(field, ig[1], s, field_weight=weight, math=math)
            assert steps.max() <= cap and (cap > 4 or steps.max() == cap)
            np.testing.assert_array_equal(steps, want_steps)
            np.testing.assert_array_equal(got, want)
