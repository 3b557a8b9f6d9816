"""Artificial conductivity's signal speed sqrt(2 |P_i - P_j| / (rho_i + rho_j))
(src/fluid_force.cpp:113-115): it vanishes between equal pressures, so the
pressures must be the particles' own, not ones worked back from a rounded
quotient; and DISPH with conductivity and no gravity agrees with the oracle."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine
from test_gpu_parity import _rel, _rms_err

pytestmark = pytest.mark.gpu


def _state(side, precision):
    """A periodic 2D lattice at rest, masses 30 % apart."""
    from sphcode_amd import _abi, ics
    n = side * side
    p, _ = ics.khi(n_low=32, n_high=45, precision=precision, sph_type=_abi.SSPH)
    p.ac_is_valid, p.ac_alpha = 1, 1.0
    grid = (np.arange(side) + 0.5) / side
    pos = np.stack(np.meshgrid(grid, grid, indexing="ij"), -1).reshape(n, 2)
    mass = (1 + 0.3 * np.random.default_rng(4).uniform(-1, 1, n)) / n
    f = dict(pos=pos, vel=np.zeros((n, 2)), mass=mass, dens=np.ones(n), ene=np.ones(n), pres=np.full(n, 2.0 / 3.0))
    assert p.kernel == _abi.WENDLAND and not p.gravity_is_valid
    return p, f


def _scale(p, d):
    """sum_j m_j c |u_i - u_j| |grad W| over the neighbours: the term at a
    signal speed of the order of the sound speed."""
    x, h, m, u = d["pos"], d["sml"], d["mass"], d["ene"]
    out = np.empty(len(m))
    for i in range(len(m)):
        dx = x - x[i]
        dx -= np.round(dx)
        q = np.sqrt((dx * dx).sum(1)) / h[i]
        t = np.maximum(1 - q, 0)
        dw = 9 / np.pi / h[i] ** 3 * 56 / 3 * q * t ** 5 * (1 + 5 * q)
        out[i] = p.ac_alpha * (m * d["sound"][i] * np.abs(u - u[i]) * dw).sum()
    return out


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("side", [24, 37])
def test_equal_pressures_conduct_nothing(gpu, side, precision):
    """u is set from the densities of a first evaluation (which do not depend
    on it) so that P = (gamma - 1) rho u is one number to three roundings of 64
    bits: a signal speed of 3e-8 of the sound speed at most, and 0 where
    pressures are compared in FP32."""
    from sphcode_amd import FP64, MIXED, GPUEngine
    p, f = _state(side, FP64 if precision == "fp64" else MIXED)
    g = GPUEngine(p)
    g.upload(f)
    g.initialize()
    f["ene"] = 0.7 / ((p.gamma - 1) * g.download(("dens",))["dens"])
    g.upload(f)
    g.initialize()
    d = g.download()
    g.close()
    assert np.ptp(d["pres"]) <= 1e-15 and np.ptp(d["ene"]) > 0.05
    err = np.abs(d["dene"]) / _scale(p, d)
    print(f"[conductivity] side={side} {precision}: heating {err.max():.1e} of the sound-speed scale", flush=True)
    assert err.max() <= 1e-6


def _sod(sph_type):
    from sphcode_amd import ics
    p, f = ics.sod(400, 50)
    p.sph_type = sph_type
    return p, f


@pytest.mark.parametrize("case", ["sod", "khi"])
def test_disph_conductivity_parity(gpu, case):
    """Without gravity, FP64, at the bars of the other parity tests."""
    from sphcode_amd import _abi, ics, GPUEngine
    p, f = _sod(_abi.DISPH) if case == "sod" else ics.khi(n_low=32, n_high=45, jitter=0.05)
    p.ac_is_valid, p.ac_alpha = 1, 1.0
    ref, g = OracleEngine(p), GPUEngine(p)
    for e in (ref, g):
        e.upload(f)
        e.initialize()
    a, b = ref.download(), g.download()
    g.close()
    for k in ("sml", "dens", "pres"):
        assert _rel(b[k], a[k]) <= 1e-9, k
    assert _rms_err(b["acc"], a["acc"]) <= 1e-8
    assert _rms_err(b["dene"], a["dene"]) <= 1e-8
