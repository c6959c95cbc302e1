"""Images read back through pinned staging against the runtime's own copies."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

import linon_amd as L
from linon_amd import scenes

pytestmark = pytest.mark.gpu


def frame(width, height):
    view = L.MainView(width, height)
    v, f, c = scenes.reference_startup_scene()
    view.update_model(v, f)
    view.update_camera(L.Camera.arcball_default(c))
    view.update_settings(L.Settings.make())
    view.set_integrator(L.Integrator.make(h_initial=0.2, adaptive=False, samples_per_ray=0, sample_steps=0))
    view.set_field("swirl")
    view.render()
    return view


# mapping images of 16 bytes a texel about the sizes where read-backs turn to chunks of 1 MiB: 3 MiB
# exactly and a row above, 4 MiB less and plus one texel, odd ones
@pytest.mark.parametrize("width, height", [(256, 768), (256, 769), (16383, 16), (1024, 256), (113, 2321), (1021, 769)])
def test_read_back_matches_the_runtimes_copy(width, height):
    """A pinned destination keeps hipMemcpy; the arrays of the read_ methods are pageable."""
    print(f"[case] {width} x {height}", flush=True)
    view = frame(width, height)
    for name in ("mapping", "final", "steps", "hit_faces"):
        got = getattr(view, f"read_{name}")()
        assert got.any()
        pinned = torch.zeros(got.nbytes, dtype=torch.uint8, pin_memory=True)
        view._check(getattr(view._lib, f"linon_read_{name}")(view._h, pinned.data_ptr(), got.nbytes))
        assert got.tobytes() == pinned.numpy().tobytes(), name


def test_read_back_from_two_threads():
    views = [frame(640, 480), frame(512, 700)]
    want = [v.read_mapping() for v in views]
    got = [None, None]

    def read(i):
        for _ in range(5):
            got[i] = views[i].read_mapping()

    threads = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g, w)


def test_two_threads_read_one_context():
    """One of them through the staging, the other meanwhile by the runtime's copy, each as it comes."""
    view = frame(1024, 700)
    want = view.read_mapping()
    got = [[], []]

    def read(i):
        for _ in range(5):
            got[i].append(view.read_mapping())

    threads = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for g in got[0] + got[1]:
        np.testing.assert_array_equal(g, want)
