"""Two particles closer than FP32's normal range, in mixed precision: their
approach enters the signal speed in full, and their force is that of FP64 at
any distance.  For the former: separation and product with the
velocity are FP32 numbers with 21 bits there, and vanish against the sums'
other terms, so 1e-5 on the time scale h / v_sig leaves room."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("sph_type", ["SSPH", "DISPH", "GSPH"])
def test_signal_speed_of_a_close_pair(gpu, dim, sph_type):
    from sphcode_amd import FP64, MIXED, GPUEngine, _abi, ics
    got = {}
    for precision in (FP64, MIXED):
        p, f = ics.rollout({1: 60, 2: 20, 3: 10}[dim], dim=dim, precision=precision)
        p.sph_type = getattr(_abi, sph_type)
        p.kernel = _abi.WENDLAND if dim > 1 else _abi.CUBIC_SPLINE
        p.periodic_is_valid = 0
        f["pos"][:2] = 0.0
        f["vel"][:2] = 0.0
        f["pos"][0, 0], f["pos"][1, 0] = -3e-39, 3e-39  # below 1.2e-38
        f["vel"][0, 0], f["vel"][1, 0] = 40.0, -40.0
        print(f"[close pair] dim={dim} {sph_type} precision={precision}", flush=True)
        g = GPUEngine(p)
        g.upload(f)
        g.initialize()
        got[precision] = g.time()[2]
        g.close()
    assert abs(got[MIXED] / got[FP64] - 1) <= 1e-5


# 1e-25: the squares are denormal; 1e-35: 1 / r times the kernel's norm is past
# FP32; 1e-42: a denormal itself; 1e-60: zero
@pytest.mark.parametrize("r", [1e-25, 1e-35, 1e-42, 1e-60])
@pytest.mark.parametrize("sph_type,kernel", [("SSPH", "CUBIC_SPLINE"), ("SSPH", "WENDLAND"), ("DISPH", "WENDLAND"), ("GSPH", "CUBIC_SPLINE")])
def test_force_of_a_close_pair(gpu, sph_type, kernel, r):
    from sphcode_amd import FP64, MIXED, GPUEngine, _abi, ics
    got = {}
    for precision in (FP64, MIXED):
        p, f = ics.rollout(10, precision=precision)
        p.sph_type = getattr(_abi, sph_type)
        p.kernel = getattr(_abi, kernel)
        p.av_use_balsara_switch = 0
        p.gsph_is_2nd_order = 0
        p.periodic_is_valid = 0
        f["pos"][:2] = 0.0
        f["pos"][0], f["pos"][1] = [-0.3 * r, 0.2 * r, 0.1 * r], [0.3 * r, -0.2 * r, -0.1 * r]
        f["vel"][:2] = 0.0
        f["vel"][0, 0], f["vel"][1, 0] = 2.0, -2.0
        print(f"[close pair] {sph_type} {kernel} r={r} precision={precision}", flush=True)
        g = GPUEngine(p)
        g.upload(f)
        g.initialize()
        got[precision] = g.download()
        g.close()
    for key in ("acc", "dene"):
        a, b = got[FP64][key], got[MIXED][key]
        assert np.isfinite(a).all() and np.isfinite(b).all(), key
        assert np.sqrt(np.mean((b - a) ** 2) / np.mean(a ** 2)) <= 1e-4, key
        assert np.max(np.abs(b[:2] - a[:2])) <= 1e-4 * np.max(np.abs(a[:2])), key
