"""Upload and download of every field: what goes up comes back bit for bit in
caller order, before and after the tree build has permuted the particles, at
sizes around a wave and over several staging buffers; absent fields come
back as zeros."""
from __future__ import annotations

import numpy as np
import pytest

from sphcode_amd import _abi, ics

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dim", [(1, 1), (63, 2), (65, 3), (4096, 2), (250007, 3)])
def test_round_trip(gpu, n, dim):
    from sphcode_amd import GPUEngine
    p, _ = ics.rollout(4, dim=dim)
    p.sph_type = _abi.GSPH
    rng = np.random.default_rng(n)
    f = {k: rng.random(_abi.field_shape(k, n, dim)) for k in _abi.ALL_FIELDS if k not in _abi.INT_FIELDS}
    f["neighbor"] = rng.integers(0, 1000, n).astype(np.int32)
    g = GPUEngine(p)
    print(f"[transfer] n={n} dim={dim}", flush=True)
    g.upload(f)
    for permuted in (False, True):
        if permuted:
            g.make_tree()
        out = g.download()
        for k in f:
            np.testing.assert_array_equal(out[k], f[k], err_msg=f"{k} permuted={permuted}")
        np.testing.assert_array_equal(out["id"], np.arange(n, dtype=np.int32))
    # fewer fields onto the same buffers: the others are zero again
    g.upload({"pos": f["pos"], "mass": f["mass"]})
    out = g.download()
    for k in _abi.ALL_FIELDS:
        if k in ("pos", "mass"):
            np.testing.assert_array_equal(out[k], f[k])
        elif k != "id":
            assert not out[k].any(), k
    g.close()
