"""Mixed precision keeps the range of FP32: densities whose square is a
denormal number, and densities whose reciprocal is one, give the forces of the
FP64 run to the mixed-precision bar (acceleration RMS 1e-4)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rms(b, a):
    return float(np.sqrt(np.mean((b - a) ** 2) / np.mean(a ** 2)))


# P / rho^2 with rho^2 denormal; 2 / (rho_i + rho_j) beyond 2^126; and both
# second-order GSPH and SSPH well inside
@pytest.mark.parametrize("sph_type,rho", [("SSPH", 2.0 ** -66), ("DISPH", 1.2 * 2.0 ** 125), ("SSPH", 2.0 ** 60),
                                          ("GSPH", 2.0 ** -56), ("GSPH", 2.0 ** 56)])
def test_densities_far_from_one(gpu, sph_type, rho):
    from sphcode_amd import FP64, MIXED, GPUEngine, _abi, ics
    got = {}
    for precision in (FP64, MIXED):
        p, f = ics.rollout(12, seed=2, precision=precision)
        p.sph_type = getattr(_abi, sph_type)
        p.gsph_is_2nd_order = 1
        f = dict(f, mass=f["mass"] * rho, dens=f["dens"] * rho, pres=f["pres"] * rho)
        g = GPUEngine(p)
        g.upload(f)
        print(f"[range] {sph_type} rho={rho:.3g} precision={precision}", flush=True)
        g.initialize()
        got[precision] = g.download()
        g.close()
    a, b = got[FP64], got[MIXED]
    assert np.isfinite(b["acc"]).all() and np.isfinite(b["dene"]).all()
    assert np.max(np.abs(b["dens"] / a["dens"] - 1)) <= 1e-5
    assert _rms(b["acc"], a["acc"]) <= 1e-4
    assert _rms(b["dene"], a["dene"]) <= 1e-4
