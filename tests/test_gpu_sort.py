"""The sort by buckets of the tree build, where it can go wrong: two to a
few particles, ragged ends of waves, key depths with many particles to a
finest cell (equal keys keep the order of their indices), and a clump that
overfills a bucket, for which the library's sort takes over.  The tree's
node count, the neighbour counts and the fields equal the oracle's to the
bars of the other parity tests, and a second engine gives the same bits."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine
from test_gpu_parity import _rel, _rms_err

pytestmark = pytest.mark.gpu


def _state(n, dim, levels, clump, seed):
    from sphcode_amd import ics
    p, _ = ics.rollout(4, dim=dim)
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1.0 / dim)))
    grid = np.stack(np.meshgrid(*[(np.arange(side) + 0.5) / side] * dim, indexing="ij"), -1).reshape(-1, dim)
    pos = grid[rng.permutation(len(grid))[:n]] + rng.uniform(-0.2, 0.2, (n, dim)) / side
    if clump:  # the same lattice, a hundredth of the size, beside a far particle
        pos = 0.3 + 0.01 * pos
        pos[n // 2] = 0.9
    p.periodic_is_valid = 0
    p.neighbor_number = 8 if n > 10 else 1
    p.tree_max_level = levels
    p.tree_leaf_particle_num = 4
    p.iterative_sml = 0 if clump or n < 10 else 1
    m = (0.01 ** dim if clump else 1.0) / n
    f = dict(pos=pos, vel=rng.normal(0.0, 0.1, (n, dim)), mass=np.full(n, m), dens=np.ones(n),
             ene=1.0 + 0.1 * rng.random(n), pres=np.full(n, 2.0 / 3.0))
    return p, f


@pytest.mark.parametrize("n,dim,levels,clump", [
    (2, 3, 20, False), (3, 2, 20, False), (63, 1, 20, False), (65, 3, 20, False), (257, 2, 20, False),
    (1025, 3, 1, False),   # eight cells in all: more than a bucket's share of equal keys
    (1025, 2, 3, False),
    (5000, 3, 2, False),   # equal keys, the buckets being the finest cells
    (511, 3, 20, True), (513, 3, 20, True), (514, 3, 20, True), (3000, 2, 20, True),
])
def test_sort_by_buckets(gpu, n, dim, levels, clump):
    from sphcode_amd import GPUEngine
    p, f = _state(n, dim, levels, clump, seed=n)
    print(f"[sort] n={n} dim={dim} levels={levels} clump={clump}", flush=True)
    engines = [OracleEngine(p), GPUEngine(p), GPUEngine(p)]
    for e in engines:
        e.upload(f)
        e.initialize()
    for _ in range(2):
        a, b, again = (e.download() for e in engines)
        assert np.array_equal(a["neighbor"], b["neighbor"])
        fin = np.isfinite(a["acc"]).all(axis=-1) if a["acc"].ndim > 1 else np.isfinite(a["acc"])
        for k in ("sml", "dens"):
            assert _rel(b[k], a[k]) <= 1e-9, k
        if fin.all():
            assert _rms_err(b["acc"], a["acc"]) <= 1e-8 and _rms_err(b["dene"], a["dene"]) <= 1e-8
        for k in ("pos", "vel", "sml", "dens", "acc", "dene"):
            assert np.array_equal(b[k], again[k], equal_nan=True), k
        for e in engines:
            e.integrate()
