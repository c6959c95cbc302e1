"""CPU checks of the rules the grid builds go by (grid.cpp and grid_build.hpp, built with g++)."""
from __future__ import annotations

import ctypes as C
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

from linon_amd import scenes

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "linon_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("grid") / "grid_shim.so"
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    f"-I{CSRC}", str(ROOT / "tests" / "host" / "grid_shim.cpp"), str(CSRC / "grid.cpp"), "-pthread",
                    "-o", str(so)], check=True)
    return C.CDLL(str(so))


def arrays(v, f):
    v = np.ascontiguousarray(v, np.float32).reshape(-1, 3)
    f = np.ascontiguousarray(f, np.uint32).reshape(-1, 3)
    return v, f, (v.ctypes.data_as(C.c_void_p), len(v), f.ctypes.data_as(C.c_void_p), len(f))


def flat(x, y=0.01):
    return np.array([[0, 0, 0], [x, 0, 0], [x, y * x, 0]], np.float32), np.array([[0, 1, 2]], np.uint32)


def test_row_masks_hold_the_longest_row(lib):
    """The cells of a dimension are counted up from rounded bounds, so a row can hold more cells than
    the resolution; the masks of a row have a bit for each."""
    longest = 0
    for x in (np.float32(0.02), *np.random.default_rng(0).uniform(1e-3, 1.0, 500)):
        v, f, args = arrays(*flat(x))
        dims = (C.c_int * 3)()
        assert lib.grid_dims(*args, 1024, dims)
        longest = max(longest, dims[0])
        assert 64 * lib.row_mask_chunks(dims[0]) >= dims[0]
        assert lib.row_mask_bytes(dims[0]) == 4 * 8 * lib.row_mask_chunks(dims[0]) <= 65536
    assert longest == 1025


def test_no_launch_has_too_many_lanes(lib):
    """A launch holds fewer than 2^32 lanes.  16 lanes a face at 2^28 faces, and a lane a reference at
    2^32 - 1 references, are as many and more; small ones get a lane each."""
    for lanes in (16 << 28, 16 * (2**32 // 3), 2**32 - 1, (1 << 22) - 1, 1 << 22):
        assert lib.stride_blocks(C.c_size_t(lanes)) * 256 < 2**32
    for lanes in (1, 16, 256, 257, 16 * 20516, (1 << 22) - 1):
        assert lanes <= lib.stride_blocks(C.c_size_t(lanes)) * 256 < lanes + 256


def test_which_grids_the_host_builds(lib):
    """Up to 2048 cells and 3072 overlap tests; a test for every cell of a face's range."""
    box = scenes.cornell_box_centered()
    for mesh, res, tiny in ((box, 4, 1), (box, 12, 1), (box, 16, 0), (box, 128, 0), (flat(1.0, 1.0), 45, 1),
                            (flat(1.0, 1.0), 46, 0), (scenes.benchmark_scene(2), 8, 1),
                            (scenes.benchmark_scene(2), 16, 0), (scenes.benchmark_scene(5), 128, 0)):
        assert lib.grid_is_tiny(*arrays(*mesh)[2], res) == tiny, (len(mesh[1]), res)
    v, f = flat(1.0, 1.0)  # three faces of 1024 cells each are the line
    assert lib.grid_is_tiny(*arrays(v, np.tile(f, (3, 1)))[2], 32) == 1
    assert lib.grid_is_tiny(*arrays(v, np.tile(f, (4, 1)))[2], 32) == 0


def test_no_memory_for_the_host_build(tmp_path):
    """Wherever in the host build memory ends, in a thread of it too, the caller gets std::bad_alloc (and
    the C entry an error); nothing is left running."""
    exe = tmp_path / "grid_memory_driver"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(ROOT / "tests" / "host" / "grid_memory_driver.cpp"), str(CSRC / "grid.cpp"), "-pthread",
                    "-o", str(exe)], check=True)
    said = []
    for k in range(4, 31):
        r = subprocess.run([str(exe), str(1 << k)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (k, r.returncode, r.stderr[-300:])
        said.append(r.stdout.strip())
    assert said[0] == "no memory" and said[-1] == "built"
