"""The adjoint's pair passes with one wave per search group, which more
particles than the other gradient tests have select (70^3: about 7,300
groups; up to 6,144 a block's four waves share one): along its own gradient
the adjoint agrees with central differences of the forward, with the step
and the bar of the 64^3 rollout's check."""
from __future__ import annotations

import numpy as np
import pytest

from sphcode_amd import ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("field", ["pos", "vel", "ene"])
def test_adjoint_one_wave_per_group(gpu, field):
    from sphcode_amd import GPUEngine
    p, f = ics.rollout(n_side=70)
    K, dt, eps = 1, 1e-3, 1e-8
    g = GPUEngine(p)

    def final(ff):
        g.upload(ff)
        g.rollout(K, dt)
        return g.download(("mass", "vel"))

    o = final(f)
    grad = dict(zip(("pos", "vel", "ene"), g.rollout_adjoint(dl_dv=2.0 * o["mass"][:, None] * o["vel"])))[field]
    d = grad / np.linalg.norm(grad)
    loss = []
    for s in (eps, -eps):
        ff = dict(f)
        ff[field] = f[field] + s * d
        if field == "pos":
            ff[field] = np.mod(ff[field], 1.0)
        o = final(ff)
        loss.append(float(np.sum(o["mass"][:, None] * o["vel"] ** 2)))
    g.close()
    fd, ad = (loss[0] - loss[1]) / (2 * eps), float(np.sum(grad * d))
    print(f"rollout 70^3 {field}: adjoint {ad:.10e} fd {fd:.10e}", flush=True)
    assert abs(ad - fd) <= 1e-4 * abs(fd)
