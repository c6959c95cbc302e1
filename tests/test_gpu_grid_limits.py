"""The device grid build where its sizes and its memory end, against the host build."""
from __future__ import annotations

import ctypes as C
import time

import numpy as np
import pytest

import linon_amd as L
from linon_amd import scenes

pytestmark = pytest.mark.gpu


def same_grids(view):
    view.set_grid_builder(L.GRID_BUILD_HOST)
    h = view.read_grid()
    view.set_grid_builder(L.GRID_BUILD_DEVICE)
    d = view.read_grid()
    for k in ("dims", "cell_start", "cell_faces", "dist", "tris"):
        np.testing.assert_array_equal(h[k], d[k], err_msg=k)
    return d


def small_faces(n, size, at, seed):
    rng = np.random.default_rng(seed)
    c = at(rng, n)[:, None, :] + size * rng.uniform(-1.0, 1.0, (n, 3, 3))
    return c.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)


def test_rows_longer_than_the_resolution():
    """Over x in [0, 0.02f] a resolution of 1024 makes 1025 cells: 17 masks of 64 cells a row.  Faces in
    the first 64 cells of some rows, in the last of others, in most none; y and z stay narrow."""
    def at(rng, n):
        x = np.where(rng.random(n) < 0.5, rng.uniform(0.0002, 0.001, n), rng.uniform(0.019, 0.0198, n))
        return np.stack([x, rng.uniform(0.0, 4e-4, n), rng.uniform(0.0, 4e-4, n)], 1)
    v, f = small_faces(60, 1e-5, at, 3)
    v = np.concatenate([v, np.array([[0, 0, 0], [0.02, 0, 0], [0.02, 1e-5, 0]], np.float32)])
    f = np.concatenate([f, [[180, 180, 180], [181, 182, 181]]]).astype(np.uint32)
    print("[case] grid build, a row of 1025 cells", flush=True)
    with L.MainView(16, 16) as view:
        view.set_grid_builder(L.GRID_BUILD_HOST)
        view.set_accel(L.ACCEL_GRID, 1024)
        view.update_model(v, f)
        d = same_grids(view)
    assert d["dims"][0] == 1025
    occupied = np.diff(d["cell_start"]).reshape(d["dims"][::-1]) > 0
    assert occupied[..., :64].any() and occupied[..., 960:].any()


def refuse(view, number):
    view._check(view._lib.linon_selftest_refuse_grid_alloc(view._h, number))


def train_one_step(view):
    view.train_surrogate(L.SurrogateConfig.make("swirl", steps=1, train_rays=2048, batch=256, lr=1e-3, h=0.01,
                                                max_steps=200, tolerance=1e-4, seed=1))


@pytest.mark.parametrize("number", range(1, 7))
def test_no_room_for_the_device_build(number):
    """Each of the build's allocations refused in turn: AUTO has the host's arrays, and the calls that
    follow know nothing of it."""
    v, f = scenes.benchmark_scene(level=3)
    print(f"[case] grid build without its allocation {number}", flush=True)
    with L.MainView(16, 16) as view:
        view.set_grid_builder(L.GRID_BUILD_HOST)
        view.update_model(v, f)
        h = view.read_grid()
        refuse(view, number)
        view.set_grid_builder(L.GRID_BUILD_AUTO)
        a = view.read_grid()
        for k in h:
            np.testing.assert_array_equal(a[k], h[k], err_msg=k)
        train_one_step(view)
        with pytest.raises(L.LinonError, match="out of memory"):
            view.set_grid_builder(L.GRID_BUILD_DEVICE)
        train_one_step(view)
        refuse(view, 0)
        view.update_model(v, f)
        same_grids(view)


def test_an_earlier_error_is_not_the_builds():
    """An error that another call on this thread left unread: the device build succeeds all the same."""
    v, f = scenes.benchmark_scene(level=2)
    print("[case] grid build after another call's error", flush=True)
    with L.MainView(16, 16) as view:
        view.set_grid_builder(L.GRID_BUILD_DEVICE)
        p = C.c_void_p()
        assert view._lib.hipMalloc(C.byref(p), C.c_size_t(1 << 50)) == 2  # hipErrorOutOfMemory
        view.update_model(v, f)
        same_grids(view)


def too_many_references():
    """Faces of half the cells of a flat 1024 x 1024 grid each, more than 2^32 references in all."""
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0]], np.float32)
    return v, np.tile(np.array([[0, 1, 2]], np.uint32), (9000, 1))


@pytest.mark.parametrize("builder, status", [(L.GRID_BUILD_AUTO, "ARGUMENT"), (L.GRID_BUILD_DEVICE, "HIP")])
def test_too_many_references_are_refused_at_once(builder, status):
    """By the device's count alone: the host would gather them all first, 34 GB."""
    v, f = too_many_references()
    print(f"[case] grid of more than 2^32 references, builder {builder}", flush=True)
    with L.MainView(16, 16) as view:
        view.set_accel(L.ACCEL_GRID, 1024)
        view.set_grid_builder(builder)
        t = time.perf_counter()
        with pytest.raises(L.LinonError, match=f"{status}.*2\\^32 face references"):
            view.update_model(v, f)
        assert time.perf_counter() - t < 30.0
        view.update_model(v, f[:1])
        same_grids(view)


@pytest.mark.parametrize("builder", [L.GRID_BUILD_AUTO, L.GRID_BUILD_DEVICE])
def test_a_refused_mesh_leaves_the_present_one(builder):
    v, f = too_many_references()
    print(f"[case] a mesh refused beside another, builder {builder}", flush=True)
    with L.MainView(32, 24) as view:
        view.set_accel(L.ACCEL_GRID, 1024)
        view.set_grid_builder(builder)
        view.update_model(v, f[:3])
        view.update_camera(L.Camera.look_at((0.3, 0.3, 1.0), (0.3, 0.3, 0.0), (0.0, 1.0, 0.0), fov_deg=60.0))
        view.set_integrator(L.Integrator.make(h_initial=0.1, adaptive=False, samples_per_ray=0, sample_steps=0))
        view.set_field("identity")
        view.render()
        want, grid = view.read_hit_faces(), view.read_grid()
        assert (want >= 0).any()
        with pytest.raises(L.LinonError, match="face references"):
            view.update_model(v, f)
        got = view.read_grid()
        for k in grid:
            np.testing.assert_array_equal(got[k], grid[k], err_msg=k)
        view.render()
        np.testing.assert_array_equal(view.read_hit_faces(), want)
        view.set_accel(L.ACCEL_GRID, 64)   # rebuilt from the context's own copy of the mesh
        view.render()
        assert (view.read_hit_faces() >= 0).any()


@pytest.mark.parametrize("offset", [0.0, 100.0, 1000.0, 1e6])
@pytest.mark.parametrize("area", [True, False])
def test_faces_far_from_the_origin_and_without_area(offset, area):
    """The short overlap test leaves the cells near an axis's threshold to the full one: more of them the
    further the mesh is from the origin, and every cell of a face that is a line or a point."""
    v, f = scenes.benchmark_scene(level=3)
    f = f.copy()
    if not area:
        f[::2, 2] = f[::2, 1]
        f[::8] = f[::8, :1]
    print(f"[case] grid build {offset} from the origin, area {area}", flush=True)
    with L.MainView(16, 16) as view:
        view.set_accel(L.ACCEL_GRID, 64)
        view.update_model((v + np.float32(offset)).astype(np.float32), f)
        d = same_grids(view)
    assert len(d["cell_faces"]) > len(f)


# lists about the line between the ranks and the sort (256), with one, two and three bytes of face id,
# and last chunks of one
@pytest.mark.parametrize("n", [250, 256, 257, 262, 300, 1025, 2049, 3073, 70001])
def test_long_lists(n):
    """n faces in a few cells about the centre, some of them reaching far, and two that span the grid."""
    rng = np.random.default_rng(n)
    v = rng.normal(size=(n, 3, 3)) * 1e-3
    v[::97] *= 100.0
    v = np.concatenate([v.reshape(-1, 3), [[-1, -1, -1], [1, 1, 1], [1, 1.01, 1], [-1, 0, 0], [1, 0, 0], [0, 1, 0]]])
    f = rng.permutation(np.arange(3 * n + 6, dtype=np.uint32).reshape(-1, 3))
    print(f"[case] {n} faces in a few cells", flush=True)
    with L.MainView(16, 16) as view:
        view.set_accel(L.ACCEL_GRID, 33)
        view.update_model(v.astype(np.float32), f)
        d = same_grids(view)
    assert np.diff(d["cell_start"]).max() > 0.98 * n
