"""FP64 pair terms divide by the separation; they do not multiply with a rounded
1/r.  Many isolated 1D pairs of one separation r, chosen so that fl(1/r) is
about half an ulp off: a product with it is off by that much in every pair,
once for each factor 1/r in the term, while a division rounds to either side.
The mean relative error of 8,192 terms against 80-bit arithmetic on the fields
that entered them is therefore near zero (a hundredth of an ulp: rounding
errors of an ulp and a half at random, over the root of their number), and may
be at most half of what one such factor gives."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

L = np.longdouble
PAIRS = 4096


def _separation():
    """r = m / 128 in (0.5, 1) whose rounded reciprocal is furthest off, and
    the relative error."""
    m = np.arange(65, 128, 2)
    r = m / 128.0
    off = (1.0 / r).astype(L) * r.astype(L) - 1
    k = int(np.argmax(np.abs(off)))
    return float(r[k]), float(off[k])


def _state(kind):
    from sphcode_amd import _abi, ics
    p, _ = ics.sod(400, 50)
    p.sph_type = _abi.SSPH
    r, off = _separation()
    rng = np.random.default_rng(3)
    x = np.empty((PAIRS, 2))
    x[:, 0] = 8.0 * np.arange(PAIRS)
    x[:, 1] = x[:, 0] + r  # exact
    v = rng.uniform(0.5, 1.5, (PAIRS, 2))
    v[:, 1] *= -1.0
    m = 1.0 + 0.1 * rng.random((PAIRS, 2))
    u = rng.uniform(1.0, 2.0, (PAIRS, 2))
    p.av_alpha = 0.0
    if kind == "viscosity":
        p.av_alpha, u = 1.0, u * 1e-40
    if kind == "conductivity":
        p.ac_is_valid, p.ac_alpha, v = 1, 1.0, 0.0 * v
    n = 2 * PAIRS
    f = dict(pos=x.reshape(n, 1), vel=v.reshape(n, 1), mass=m.reshape(n), dens=np.full(n, 0.7 / r), ene=u.reshape(n),
             pres=np.ones(n))
    return p, f, off


def _exact(p, d):
    """du/dt of every particle from its pair, in 80 bits (src/fluid_force.cpp:59-116)."""
    def both(k):
        a = d[k].reshape(PAIRS, 2).astype(L)
        return a.reshape(-1), a[:, ::-1].reshape(-1)
    (xi, xj), (vi, vj), (hi, hj), (ri, rj), (pi, pj) = (both(k) for k in ("pos", "vel", "sml", "dens", "pres"))
    (mi, mj), (ui, uj), (ci, cj), (gi, _), (ai, aj), (bi, bj) = (both(k) for k in ("mass", "ene", "sound", "gradh", "alpha", "balsara"))
    d1, v = xi - xj, vi - vj
    r = np.abs(d1)

    def grad(h):
        q = 2 * r / h
        a, b = np.maximum(2 - q, 0), np.maximum(1 - q, 0)
        return -L(2.0 / 3.0) * (2 / h) ** 2 / r * (L(0.75) * a * a - 3 * b * b) * d1
    dwi, dwj = grad(hi), grad(hj)
    dw = (dwi + dwj) / 2
    out = mj * pi / ri ** 2 * gi * v * dwi
    w = np.minimum(v * d1, 0) / r
    visc = -(bi + bj) / 2 * (ai + aj) / 2 * (ci + cj - 3 * w) * w * (2 / (ri + rj))
    out += mj * visc / 4 * 2 * v * dw / 2
    if p.ac_is_valid:
        out += L(p.ac_alpha) * mj * np.sqrt(2 * np.abs(pi - pj) / (ri + rj)) * (ui - uj) * dw * d1 / r
    return out


@pytest.mark.parametrize("kind", ["pressure", "viscosity", "conductivity"])
def test_pair_terms_divide(gpu, kind):
    from sphcode_amd import GPUEngine
    p, f, off = _state(kind)
    g = GPUEngine(p)
    g.upload(f)
    g.initialize()
    d = g.download()
    g.close()
    assert (d["neighbor"] == 2).all()
    want = _exact(p, d)
    rel = (d["dene"].astype(L) - want) / want
    print(f"[quotients] {kind}: mean {float(rel.mean()):.3e} largest {float(np.abs(rel).max()):.3e}, 1/r off by {off:.3e}", flush=True)
    assert abs(float(rel.mean())) <= 0.5 * abs(off)
