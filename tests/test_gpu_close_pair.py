"""Two particles closer than FP32's normal range, in mixed precision: their
approach enters the signal speed in full.  Separation and product with the
velocity are FP32 numbers with 21 bits there, and vanish against the sums'
other terms, so 1e-5 on the time scale h / v_sig leaves room."""
from __future__ import annotations

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
