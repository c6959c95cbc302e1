"""Builds liblinon_hip.so (gfx950) in-tree with hipcc.

Usage: python -m linon_amd.build [--jobs N]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
BUILD = ROOT / "_build" / "linon_hip"
LIB = PKG / "liblinon_hip.so"
ARCH = "gfx950"

# Packed-FP32 instructions are disabled for all device code (they are not trusted on the
# target machines); the host pass warns that it does not know the feature, harmlessly.
DEVICE_FLAGS = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
COMMON = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall", "-Wno-unused-result",
          f"-I{ROOT / 'include'}", f"-I{CSRC}"]

SOURCES = ["kernels.hip", "surrogate.hip", "grid_build.hip", "noalloc.hip", "context.cpp", "grid.cpp", "jit.cpp", "wgsl.cpp", "batch.cpp", "readback.cpp", "surrogate.cpp"]
# The ray-cast and surrogate kernels are compiled a second time with the accuracy WGSL itself
# specifies (approximate division and sqrt, hardware transcendentals) into namespace
# linon_wgslmath; linon_set_math chooses between the two builds per field.
WGSL_MATH_FLAGS = ["-DLINON_FAST_MATH", "-DLINON_KERNEL_NS=linon_wgslmath",
                   "-fno-hip-fp32-correctly-rounded-divide-sqrt", "-fgpu-approx-transcendentals"]
WGSL_MATH_SOURCES = ["kernels.hip", "surrogate.hip"]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc"):
        if cand and Path(cand).exists():
            return cand
    return "hipcc"


def _compile(src: Path, obj: Path, extra: tuple = ()) -> tuple[str, int, str]:
    cmd = [hipcc(), *COMMON, *DEVICE_FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    if src.suffix == ".hip":
        cmd[1:1] = ["-x", "hip"]
    p = subprocess.run(cmd, capture_output=True, text=True)
    out = "\n".join(l for l in (p.stdout + p.stderr).splitlines() if "packed-fp32-ops" not in l)
    return " ".join(cmd), p.returncode, out


def generate_embedded_source(dst: Path) -> None:
    """Embeds the device headers as one string so hiprtc can compile user fields."""
    parts = []
    dev = CSRC / "device"
    for name in ("params.hpp", "wgsl_lib.hpp", "raycast.hpp"):
        text = (dev / name).read_text()
        text = "\n".join(l for l in text.splitlines()
                         if not l.startswith('#include "') and l.strip() != "#pragma once")
        parts.append(f"// ---- {name}\n{text}\n")
    body = "".join(parts)
    delim = "LINONSRC"
    assert f"){delim}\"" not in body
    dst.write_text(
        "// generated by linon_amd/build.py from csrc/device/*.hpp\n"
        f'extern "C" const char linon_device_source[] = R"{delim}(\n{body}){delim}";\n')


def build(jobs: int = 8, verbose: bool = False) -> Path:
    BUILD.mkdir(parents=True, exist_ok=True)
    gen = BUILD / "embedded_source.cpp"
    generate_embedded_source(gen)
    srcs = [CSRC / s for s in SOURCES if (CSRC / s).exists()] + [gen]
    objs = [BUILD / (s.name + ".o") for s in srcs]
    extras = [()] * len(srcs)
    for name in WGSL_MATH_SOURCES:
        srcs.append(CSRC / name)
        objs.append(BUILD / (name + ".wgslmath.o"))
        extras.append(tuple(WGSL_MATH_FLAGS))
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        results = list(ex.map(_compile, srcs, objs, extras))
    failed = False
    for (cmd, rc, out), s in zip(results, srcs):
        if verbose or rc != 0:
            print(f"[build] {s.name}: rc={rc}\n{cmd}\n{out}", file=sys.stderr)
        failed |= rc != 0
    if failed:
        raise RuntimeError("liblinon_hip build failed")
    tmp = LIB.with_suffix(".so.tmp")
    link = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs),
            "-lhiprtc", "-Wl,-rpath,/opt/rocm/lib"]
    p = subprocess.run(link, capture_output=True, text=True)
    if p.returncode != 0:
        raise RuntimeError("link failed:\n" + " ".join(link) + "\n" + p.stdout + p.stderr)
    os.replace(tmp, LIB)
    return LIB


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=8)
    ap.add_argument("-v", "--verbose", action="store_true")
    a = ap.parse_args()
    print(build(a.jobs, a.verbose))


if __name__ == "__main__":
    main()
