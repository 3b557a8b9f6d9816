"""A particle that has lost its position (NaN) interacts with none, and all the
others go on as if it were not there: the same neighbour sets and fields as
the oracle's, for a NaN in any axis and in the first slots of the tree order
(a NaN compares as the lower half of every cell), with the periodic box and
without, with one wave per search group and with four."""
from __future__ import annotations

import numpy as np
import pytest

from _oracle import OracleEngine
from test_gpu_parity import _rel, _rms_err
from test_gpu_search import _state

pytestmark = pytest.mark.gpu


# the last two have particles enough that a wave takes a group by itself, in
# the search (3D) and in the pair passes too (2D)
@pytest.mark.parametrize("n,dim,periodic,lost", [
    (5000, 3, False, [(0, 7)]), (5000, 3, True, [(0, 7)]), (5000, 3, True, [(1, 7), (2, 4999)]),
    (6001, 2, True, [(0, 0), (1, 1), (1, 3000)]), (6001, 2, False, [(1, 6000)]), (4000, 1, True, [(0, 1234)]),
    (120_001, 3, True, [(0, 11)]), (420_001, 2, True, [(0, 11)]),
])
def test_lost_particle(gpu, n, dim, periodic, lost):
    from sphcode_amd import GPUEngine
    p, f = _state(n, dim, periodic, 16 if dim > 1 else 4, 8, seed=n)
    assert n > max(8 * 20, 48) * p.neighbor_number  # a box near everything would pass the candidates' slots
    for axis, i in lost:
        f["pos"][i, axis] = np.nan
    gone = np.array(sorted({i for _, i in lost}))
    rest = np.setdiff1d(np.arange(n), gone)
    ref, g = OracleEngine(p), GPUEngine(p)
    print(f"[lost] n={n} dim={dim} periodic={periodic} lost={lost}", flush=True)
    for e in (ref, g):
        e.upload(f)
        e.initialize()
    for step in range(3):
        a, b = ref.download(), g.download()
        assert np.array_equal(a["neighbor"], b["neighbor"]), step
        assert not a["neighbor"][gone].any()
        for k in ("sml", "dens", "pres"):
            assert _rel(b[k][rest], a[k][rest]) <= 1e-9, k
        assert _rms_err(b["acc"][rest], a["acc"][rest]) <= 1e-8 and _rms_err(b["dene"][rest], a["dene"][rest]) <= 1e-8
        for e in (ref, g):
            e.integrate(1e-4)
    g.close()
