"""Pairs that sit on the cut across a periodic face.  On a 1D lattice with a
cubic spline and four neighbours, h is two spacings to round-off, so that
which of the second neighbours counts is decided by the last bits of the pair's
minimum image: |(x_i - x_j) + L| as the reference takes it, not the distance to
a coordinate that was moved by L first (include/periodic.hpp:34-59).  Without
the Newton solve the search radius, h and the cut are one number, which is read
back here; counts and sets are then exact."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

REACH = 4  # lattice neighbours looked at to each side


def _lattice(n, gap):
    from sphcode_amd import ics
    p, _ = ics.sod(400, 50)
    p.periodic_is_valid, p.iterative_sml, p.neighbor_number = 1, 0, 4
    p.range_min[0], p.range_max[0] = 0.0, 1.0
    p.tree_leaf_particle_num = 3
    x = (np.arange(n) + 0.5) / n
    if gap:  # a shifted lattice, so that the faces cut it elsewhere
        x = np.mod(x + 0.31, 1.0)
        x.sort()
    f = dict(pos=x[:, None], vel=np.zeros((n, 1)), mass=np.full(n, 1.0 / n), dens=np.ones(n), ene=np.ones(n),
             pres=np.full(n, 0.4))
    return p, f


def _distance(x, o):
    """Minimum-image distance from every particle to its o-th neighbour."""
    d = x - np.roll(x, -o)
    d2, d3 = d + 1.0, d - 1.0
    a1, a2, a3 = np.abs(d), np.abs(d2), np.abs(d3)
    r = np.where((a1 <= a2) & (a1 <= a3), d, np.where((a2 <= a3) & (a2 <= a1), d2, d3))
    return np.sqrt(r * r)


def _expected(x, h):
    """Per particle: neighbours with r < h_i (itself among them), and the
    partners with r < max(h_i, h_j)."""
    n = len(x)
    count, partners = np.ones(n, int), [[] for _ in range(n)]
    pairs = 0
    for o in [k for k in range(-REACH, REACH + 1) if k]:
        r = _distance(x, o)
        assert abs(o) < REACH or not (r < np.maximum(h, np.roll(h, -o))).any()
        count += (r < h) & (r * r < h * h)
        near = r < np.maximum(h, np.roll(h, -o))
        pairs += int(near.sum())
        if n < 2000:
            for i in np.nonzero(near)[0]:
                partners[i].append((i + o) % n)
    return count, partners, pairs


@pytest.mark.parametrize("n,gap", [(57, False), (90, False), (90, True), (1000, False), (1001, True),
                                   (400_003, False)])  # the last with a wave to each group
def test_cut_across_face(gpu, n, gap):
    from sphcode_amd import GPUEngine
    p, f = _lattice(n, gap)
    g = GPUEngine(p, stats=True)
    g.set_record_sets(n < 2000)
    g.upload(f)
    print(f"[cut] n={n} gap={gap}", flush=True)
    g.initialize()
    for step in range(2):
        d = g.download(("pos", "sml", "neighbor"))
        x = d["pos"][:, 0]
        assert np.array_equal(x, f["pos"][:, 0])
        count, partners, pairs = _expected(x, d["sml"])
        assert np.array_equal(d["neighbor"], count), f"step {step}: {np.nonzero(d['neighbor'] != count)[0]}"
        assert g.stats()["force_pairs"] == pairs
        if n < 2000:
            got = g.neighbor_sets(1)
            bad = [i for i in range(n) if sorted(got[i]) != sorted(partners[i])]
            assert not bad, f"step {step}: force sets of {bad}"
        g.reset_stats()
        g.integrate(1e-30)  # nothing moves; the searches are one now
    g.close()
