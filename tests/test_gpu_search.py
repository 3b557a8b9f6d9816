"""The box search at the edges of its chunks (32 particles), groups (64) and
second- and third-level boxes (2,048 and 131,072): the recorded gather and
force sets equal the oracle's, per particle, and the summed fields agree
to the FP64 bars of the other parity tests.  The periodic states include
ones whose search radius spans the box, where every pair takes its own
minimum image."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine
from test_gpu_parity import _check_sets, _rel, _rms_err

pytestmark = pytest.mark.gpu


def _state(n, dim, periodic, neighbours, leaf, seed):
    from sphcode_amd import ics
    p, _ = ics.rollout(4, dim=dim)
    rng = np.random.default_rng(seed)
    # a lattice of n sites with jitter, so that no two particles coincide
    side = int(np.ceil(n ** (1.0 / dim)))
    grid = np.stack(np.meshgrid(*[(np.arange(side) + 0.5) / side] * dim, indexing="ij"), -1).reshape(-1, dim)
    pos = np.mod(grid[rng.permutation(len(grid))[:n]] + rng.uniform(-0.2, 0.2, (n, dim)) / side, 1.0)
    p.periodic_is_valid = 1 if periodic else 0
    p.neighbor_number = neighbours
    p.tree_leaf_particle_num = leaf
    p.neighbor_capacity = max(4 * n, 64) if n < 300 else 0
    f = dict(pos=pos, vel=rng.normal(0.0, 0.1, (n, dim)), mass=np.full(n, 1.0 / n), dens=np.ones(n),
             ene=1.0 + 0.1 * rng.random(n), pres=np.full(n, 2.0 / 3.0))
    return p, f


@pytest.mark.parametrize("n,dim,periodic,neighbours,leaf", [
    (2, 3, False, 1, 1), (31, 3, False, 8, 1), (33, 3, True, 8, 4), (64, 2, True, 12, 1), (65, 3, False, 16, 32),
    (65, 3, True, 40, 1),       # the search radius spans the periodic box
    (100, 2, True, 60, 8),      # and in 2D
    (63, 1, True, 4, 1), (2047, 3, True, 32, 8), (2049, 3, True, 32, 1), (4097, 2, True, 24, 3),
    (131073, 3, True, 20, 16),  # two third-level boxes
])
def test_search_sets_at_edges(gpu, n, dim, periodic, neighbours, leaf):
    from sphcode_amd import GPUEngine
    p, f = _state(n, dim, periodic, neighbours, leaf, seed=n)
    ref, g = OracleEngine(p), GPUEngine(p)
    print(f"[search] n={n} dim={dim} periodic={periodic}", flush=True)
    big = n > 10000
    for e in (ref, g):
        e.set_record_sets(not big)
        e.upload(f)
        e.initialize()
    if not big:
        _check_sets(ref, g, f"n={n}", p)
    for _ in range(2):
        a, b = ref.download(), g.download()
        assert np.array_equal(a["neighbor"], b["neighbor"])
        for k in ("sml", "dens", "pres"):
            assert _rel(b[k], a[k]) <= 1e-9, k
        assert _rms_err(b["acc"], a["acc"]) <= 1e-8 and _rms_err(b["dene"], a["dene"]) <= 1e-8
        for e in (ref, g):
            e.integrate()
        if not big:
            # the combined search, whose radii are the larger of the pair's
            for x, y in zip(ref.neighbor_sets(0), g.neighbor_sets(0)):
                assert np.array_equal(x, y)
    g.close()


@pytest.mark.parametrize("dim,periodic", [(1, False), (2, False), (3, False), (3, True)])
def test_boxes_far_from_zero(gpu, dim, periodic):
    """A domain far from zero: the FP32 boxes are as tight as near zero (the
    same number is tested, within the root cube's rounding) and the
    neighbour counts are the same.  Positions are multiples of 2^-26, so that
    the shift by 2^26 is exact."""
    from sphcode_amd import GPUEngine
    n, shift = 9000, 2.0 ** 26
    p, f = _state(n, dim, periodic, 16 if dim > 1 else 6, 8, seed=dim)
    f["pos"] = np.round(f["pos"] * 2.0 ** 26) / 2.0 ** 26
    got = []
    for off in (0.0, shift):
        if periodic:
            for k in range(dim):
                p.range_min[k], p.range_max[k] = off, off + 1.0
        g = GPUEngine(p, stats=True)
        g.upload(dict(f, pos=f["pos"] + off))
        print(f"[search] dim={dim} periodic={periodic} shift={off}", flush=True)
        g.initialize()
        nb = g.download()["neighbor"]
        g.integrate()
        got.append((g.stats()["search_nodes"], nb))
        g.close()
    assert np.array_equal(got[0][1], got[1][1])
    assert got[1][0] <= 1.05 * got[0][0]
