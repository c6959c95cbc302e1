"""CPU checks of the staged read-back (readback.cpp, built with g++ over HIP calls that copy host
memory)."""
from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
CSRC = ROOT / "linon_amd" / "csrc"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    exe = tmp_path_factory.mktemp("readback") / "readback_driver"
    subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", f"-I{CSRC}",
                    str(ROOT / "tests" / "host" / "readback_driver.cpp"), str(CSRC / "readback.cpp"), "-pthread",
                    "-o", str(exe)], check=True)

    def run(*args):
        r = subprocess.run([str(exe), *map(str, args)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, (r.returncode, r.stderr[-500:])
        return {k: int(v) for k, v in re.findall(r"(\w+) (\d+)", r.stdout)}
    return run


def test_no_memory_for_a_thread(driver):
    """Where no thread can be made, the calling one copies everything; nothing is thrown."""
    r = driver("no_memory")
    assert r["error"] == 0 and r["equal"] and r["staged"] == 11


def test_a_failed_transfer_is_reported(driver):
    r = driver("fail")
    assert r["error"] != 0 and not r["equal"]


def test_no_pinned_memory(driver):
    r = driver("no_pinned")
    assert r["error"] == 0 and r["equal"] and (r["staged"], r["plain"]) == (0, 2)


@pytest.mark.parametrize("size, staged", [((4 << 20) - 1, False), (4 << 20, True)])
def test_copies_from_4_mib_are_staged(driver, size, staged):
    r = driver("size", size)
    assert r["error"] == 0 and r["equal"] and (r["staged"] > 0, r["plain"] > 0) == (staged, not staged)


def test_a_second_reader_has_the_runtimes_copy(driver):
    """Two threads read one context: the second does not wait for the first one's slots."""
    r = driver("second")
    assert r["error"] == 0 and r["equal"] and (r["staged"], r["plain"]) == (11, 1)
