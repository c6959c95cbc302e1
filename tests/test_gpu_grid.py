"""GPU: the device build of the uniform grid (count / scan / fill / per-cell sort / distance
field kernels) against the host build, array for array, and the frames each grid renders."""
from __future__ import annotations

import numpy as np
import pytest

import linon_amd as L
from linon_amd import configs, scenes

pytestmark = pytest.mark.gpu


def _grid(view, builder):
    view.set_grid_builder(builder)
    return view.read_grid()


# ico8 is the 4K stress scene: the Cornell box plus the level-8 icosphere (1,310,756 faces) at
# the resolution the context picks for it
@pytest.mark.parametrize("mesh,res", [("cornell", 0), ("ico3", 0), ("ico6", 128), ("ico6", 256), ("ico8", 0),
                                      ("empty", 0)])
def test_device_grid_equals_host_grid(mesh, res):
    if mesh == "cornell":
        v, f = scenes.cornell_box_centered()
    elif mesh == "empty":
        v, f = np.zeros((0, 3), np.float32), np.zeros((0, 3), np.uint32)
    else:
        v, f = scenes.benchmark_scene(level=int(mesh[3:]))
    print(f"[case] grid build {mesh} ({len(f)} faces) res={res}", flush=True)
    view = L.MainView(64, 48)
    try:
        view.set_accel(L.ACCEL_GRID, res)
        view.set_grid_builder(L.GRID_BUILD_HOST)
        view.update_model(v, f)
        h = view.read_grid()
        d = _grid(view, L.GRID_BUILD_DEVICE)
        assert np.array_equal(h["dims"], d["dims"])
        assert np.array_equal(h["cell_start"], d["cell_start"])
        assert np.array_equal(h["cell_faces"], d["cell_faces"])
        assert np.array_equal(h["dist"], d["dist"])
        assert np.array_equal(h["tris"], d["tris"])
    finally:
        view.close()


def test_device_grid_renders_the_same_frame():
    wl = configs.OVERLAY_1080P
    v, f = scenes.benchmark_scene(level=4)
    view = L.MainView(96, 64)
    try:
        view.update_camera(wl.camera())
        view.update_settings(wl.settings())
        view.set_integrator(wl.integrator())
        view.set_field("lens")
        frames = []
        for builder in (L.GRID_BUILD_HOST, L.GRID_BUILD_DEVICE):
            print(f"[case] grid render builder={builder}", flush=True)
            view.set_grid_builder(builder)
            view.update_model(v, f)
            view.render()
            frames.append(view.read_frame())
        a, b = frames
        assert (a.hit_faces >= 0).mean() > 0.05
        assert np.array_equal(a.hit_faces, b.hit_faces)
        assert np.array_equal(a.mapping, b.mapping)
        assert np.array_equal(a.final, b.final)
    finally:
        view.close()


def _lists(v, f, res=0):
    """The grid of (v, f) from either builder, and from the automatic choice."""
    out = []
    with L.MainView(16, 16) as view:
        view.set_accel(L.ACCEL_GRID, res)
        view.update_model(v, f)
        for b in (L.GRID_BUILD_HOST, L.GRID_BUILD_DEVICE, L.GRID_BUILD_AUTO):
            out.append(_grid(view, b))
    return out


@pytest.mark.parametrize("shape", ["wall", "crowd", "slab", "wide_rows", "one"])
def test_device_grid_edges(shape):
    """Faces and grids at the builder's edges: one face over most cells (spread over the blocks),
    hundreds of faces in one cell (long lists to rank), a flat mesh (one cell layer), rows longer
    than eight 64-cell chunks with empty stretches beyond the distance's cap of 255, one face."""
    rng = np.random.default_rng(11)
    res = 0
    if shape == "wall":
        v = np.array([[-1, -1, -1], [1, 1, -0.9], [-1, 1, 1], [0.9, -1, 1]], np.float32)
        f = np.array([[0, 1, 2], [1, 2, 3], [0, 3, 2]], np.uint32)
    elif shape == "crowd":  # 700 small faces inside one cell of a grid that another face stretches
        v = np.concatenate([rng.uniform(0.0, 1e-3, (2100, 3)), [[4, 4, 4], [4, 3.9, 4], [3.9, 4, 4]]]).astype(np.float32)
        f = np.arange(2103, dtype=np.uint32).reshape(-1, 3)[rng.permutation(701)]
    elif shape == "slab":
        v = np.concatenate([rng.uniform(-1, 1, (300, 2)), np.zeros((300, 1))], 1).astype(np.float32)
        f = rng.integers(0, 300, (257, 3)).astype(np.uint32)
    elif shape == "wide_rows":
        v = np.array([[0, 0, 0], [0.01, 0, 0], [0, 0.01, 0.01], [1, 0.02, 0.03], [0.99, 0, 0.01], [1, 0, 0]], np.float32)
        f = np.arange(6, dtype=np.uint32).reshape(2, 3)
        res = 700
    else:
        v, f = np.eye(3, dtype=np.float32), np.array([[0, 1, 2]], np.uint32)
    print(f"[case] grid edges {shape} ({len(f)} faces)", flush=True)
    h, d, auto = _lists(v, f, res)
    for k in ("dims", "cell_start", "cell_faces", "dist", "tris"):
        assert np.array_equal(h[k], d[k]) and np.array_equal(h[k], auto[k]), k
