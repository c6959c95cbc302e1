"""GPU: the lists of a surrogate frame (rays that entered, RK4 fallback, re-judged rays) at image
sizes around their tiles and blocks."""
from __future__ import annotations

import numpy as np
import pytest

import linon_amd as L
from linon_amd import configs

from gpu_common import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W,H", [(2, 2), (9, 7), (64, 16), (65, 33), (131, 97)])
@pytest.mark.parametrize("field", ["warp", "lens"])   # warp accepts most rays, lens lists all for RK4
def test_frame_lists(W, H, field):
    """Every entered ray is accepted or on one of the two RK4 lists exactly once: the counts add up,
    the mask agrees with them, and each texel without the mask holds the plain frame's exit (an
    entry lost or written twice would leave another ray's, or none: the parity bound 1e-4)."""
    wl = configs.OVERLAY_1080P
    with L.MainView(W, H) as view:
        view.update_model(np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32))
        view.update_camera(wl.camera())
        view.update_settings(wl.settings())
        view.load_surrogate(configs.saved_surrogate(field, wl))
        view.set_integrator(L.Integrator.make(h_initial=wl.h, t_max=1e30, adaptive=False, max_steps=wl.max_steps,
                                              mode=L.MODE_ESCAPE, escape_radius=2.0, samples_per_ray=0,
                                              sample_steps=0, need_mapping=True, clip_exit=True))
        view.set_field(field)
        print(f"[case] surrogate lists {field} {W}x{H}", flush=True)
        view.render()
        plain = view.read_mapping()
        view.render_surrogate()
        st = view.surrogate_stats()
        got, acc = view.read_mapping(), view.read_surrogate_accepted()
    assert st["accepted"] + st["conf_fallback"] + st["lyapunov_fallback"] == st["entered"] <= W * H
    assert st["accepted"] == int(acc.sum()) and st["rejudged"] <= st["accepted"]
    assert (rel_err(got, plain)[~acc] <= 1e-4).all()
