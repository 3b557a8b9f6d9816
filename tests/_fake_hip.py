"""Builds a host program from the library's own sources over a HIP runtime that
needs no GPU (fake_hip.cpp)."""
from __future__ import annotations

import concurrent.futures as cf
import pathlib
import subprocess

from sphcode_amd import build

HERE = pathlib.Path(__file__).resolve().parent


def _compile(src: pathlib.Path, out: pathlib.Path) -> pathlib.Path:
    cmd = [build.HIPCC, "--offload-host-only", "-std=c++17", "-O1", "-fPIC", "-I", str(build.ROOT / "include"),
           "-x", "hip", "-c", str(src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, f"{' '.join(cmd)}\n{r.stderr}"
    return out


def program(driver: str, where: pathlib.Path, without=()) -> pathlib.Path:
    """`driver` with the library's sources, except those that it includes itself."""
    srcs = [build.SRC / s for s in build.SOURCES if s not in without] + [HERE / "fake_hip.cpp", HERE / driver]
    with cf.ThreadPoolExecutor(8) as ex:
        objs = list(ex.map(lambda s: _compile(s, where / (s.stem + ".o")), srcs))
    exe = where / "program"
    # (the device code that the host objects refer to is left out)
    r = subprocess.run([build.CXX, "-o", str(exe), *map(str, objs), "-lpthread", "-Wl,--unresolved-symbols=ignore-all"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return exe
