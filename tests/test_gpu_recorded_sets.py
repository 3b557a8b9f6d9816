"""The recorded force sets are as large, particle by particle, as the number of
pairs that the force pass itself has summed (sphgpu_neighbor_sets refuses
others), and are the oracle's, over the forms that the pass takes: one and four waves to a group, periodic images that are the
candidate's own, shifted or each pair's, one to three dimensions, every
formulation, FP64 and mixed.  Likewise the pre-interaction counts as many pairs
as the oracle's neighbour numbers add up to."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine
from test_gpu_search import _state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n,dim,periodic,neighbours,sph_type", [
    (65, 3, True, 40, "SSPH"),   # every pair takes its own image
    (100, 2, True, 60, "DISPH"),
    (63, 1, True, 4, "SSPH"), (2049, 3, True, 32, "DISPH"), (4097, 2, True, 24, "GSPH"), (2047, 3, False, 32, "GSPH"),
    (90_001, 1, True, 4, "SSPH"),
    (400_001, 2, True, 12, "DISPH"),  # one wave to a group
])
def test_recorded_force_sets(gpu, n, dim, periodic, neighbours, sph_type, precision):
    from sphcode_amd import FP64, MIXED, GPUEngine, _abi
    p, f = _state(n, dim, periodic, neighbours, 8, seed=n)
    p.sph_type = getattr(_abi, sph_type)
    p.gsph_is_2nd_order = 1
    ref = OracleEngine(p)
    p.precision = FP64 if precision == "fp64" else MIXED
    g = GPUEngine(p, stats=True)
    print(f"[record] n={n} dim={dim} periodic={periodic} {sph_type} {precision}", flush=True)
    for e in (ref, g):
        e.set_record_sets(True)
        e.upload(f)
    for step in range(2):
        before = (ref.stats(), g.stats())
        for e in (ref, g):
            e.initialize() if step == 0 else e.integrate(1e-5)
        a, b = ({k: e.stats()[k] - s[k] for k in ("force_pairs", "gather_pairs")} for e, s in zip((ref, g), before))
        offs, members = g.neighbor_sets_packed(1)
        assert offs[-1] == b["force_pairs"]
        nb = g.download(("neighbor",))["neighbor"]
        assert nb.sum() == b["gather_pairs"]
        roffs, rmembers = ref.neighbor_sets_packed(1)
        if precision == "fp64":
            assert a == b
            assert np.array_equal(offs, roffs) and np.array_equal(members[:offs[-1]], rmembers[:roffs[-1]])
        else:
            # a pair at the very edge may fall to either side (h of FP32 sums, 1e-7 off)
            assert abs(a["force_pairs"] - b["force_pairs"]) <= 1e-5 * a["force_pairs"] + 1
    g.close()
