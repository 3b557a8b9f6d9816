"""Cells that span slices of 2,048 nodes, at the edges of a slice and on both
sides of the line between one workgroup and a launch for each level: geometry
and counts equal the oracle's, the moments are sums in the same order whichever
way they were taken (the first build of a state decides by an estimate, the
second by the first's nodes), and within n * 2^-52 of the oracle's."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine

pytestmark = pytest.mark.gpu

SLICE = 2048
LINE = 2_000_000  # nodes


def _params(dim, leaf):
    from sphcode_amd import ics
    p, _ = ics.rollout(4, dim=dim)
    p.periodic_is_valid = 0
    p.tree_leaf_particle_num = leaf
    return p


def _compare(p, pos, mass):
    from sphcode_amd import GPUEngine
    n, dim = pos.shape
    f = dict(pos=pos, vel=np.zeros((n, dim)), mass=mass, dens=np.ones(n), ene=np.ones(n), pres=np.ones(n))
    ref, g = OracleEngine(p), GPUEngine(p)
    ref.upload(f)
    ref.make_tree()
    a = ref.tree_info()
    g.upload(f)
    got = []
    for _ in range(2):
        g.make_tree()
        got.append(g.tree_info())
    g.close()
    eps = n * 2.0 ** -52
    for b in got:
        assert a["num_nodes"] == b["num_nodes"]
        assert np.array_equal(a["level"], b["level"]) and np.array_equal(a["count"][1:], b["count"][1:])
        assert np.array_equal(a["edge"], b["edge"]) and np.array_equal(a["center"], b["center"])
        assert np.allclose(a["mass"], b["mass"], rtol=eps, atol=0)
        assert np.max(np.abs(a["com"][1:] - b["com"][1:])) <= 2 * eps * np.abs(pos).max()
    assert np.array_equal(got[0]["mass"], got[1]["mass"]) and np.array_equal(got[0]["com"], got[1]["com"])
    return a["num_nodes"]


def _with_nodes(p, want, dim, rng):
    """A state whose tree has exactly `want` nodes."""
    pos = rng.random((want, dim))
    ref = OracleEngine(p)

    def count(k):
        x = pos[:k]
        ref.upload(dict(pos=x, vel=0 * x, mass=np.ones(k), dens=np.ones(k), ene=np.ones(k), pres=np.ones(k)))
        ref.make_tree()
        return ref.tree_info()["num_nodes"]

    lo, hi = 2, want  # (more particles: a few nodes more each time, seldom fewer)
    while hi - lo > 8:
        mid = (lo + hi) // 2
        lo, hi = (mid, hi) if count(mid) < want else (lo, mid)
    for k in range(max(2, lo - 60), min(hi + 60, want + 1)):
        if count(k) == want:
            return pos[:k]
    return None


@pytest.mark.parametrize("nodes", [SLICE - 1, SLICE, SLICE + 1, 2 * SLICE, 2 * SLICE + 1])
@pytest.mark.parametrize("dim", [2, 3])
def test_nodes_at_slice_edges(gpu, nodes, dim):
    p = _params(dim, 2)
    for seed in range(20):
        rng = np.random.default_rng(seed)
        pos = _with_nodes(p, nodes, dim, rng)
        if pos is not None:
            break
    print(f"[span] {len(pos)} particles for {nodes} nodes, dim={dim}", flush=True)
    assert _compare(p, pos, rng.random(len(pos)) + 0.5) == nodes


def test_both_sides_of_the_line(gpu):
    """A lattice whose nodes are fewer than the line while the estimate before
    the first build is above it."""
    p = _params(3, 1)
    n = 1_560_000
    side = int(np.ceil(n ** (1 / 3)))
    rng = np.random.default_rng(5)
    pos = np.stack(np.meshgrid(*[(np.arange(side) + 0.5) / side] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    pos = pos + rng.uniform(-0.2, 0.2, pos.shape) / side
    print(f"[span] n={n}", flush=True)
    nodes = _compare(p, pos, rng.random(n) + 0.5)
    assert nodes < LINE < 1.3 * n
