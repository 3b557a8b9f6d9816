"""The time step's reduction at the edges of its launches: one block up to
4,096 particles, then a block per 1,024 up to one per CU.  A minimum is
exact and each term takes the same correctly rounded operations, so the
result equals numpy's to the bit; particles at rest, NaN and infinite
entries count as they do one by one."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(h, acc, hvs, sound, force):
    # |a|^2 is summed with fused multiply-adds on the device: exact here, as
    # the components are small integers
    a = np.sqrt((acc ** 2).sum(0))
    with np.errstate(all="ignore"):
        d = force * np.sqrt(h / a)
    d = d[(a > 0) & ~np.isnan(d)]
    return min(sound * hvs, d.min() if len(d) else 1.7976931348623157e308)


@pytest.mark.parametrize("n", [1, 63, 1024, 1025, 4095, 4096, 4097, 5121, 262144, 262145, 600001])
@pytest.mark.parametrize("dim", [1, 3])
def test_timestep_sizes(gpu, n, dim):
    import torch
    from sphcode_amd import library
    fn = library()[0].sphgpu_timestep_noalloc
    fn.restype = C.c_int
    fn.argtypes = [C.c_int, C.c_int64] + [C.c_void_p] * 5 + [C.c_double] * 2 + [C.c_void_p] * 2
    rng = np.random.default_rng(n)
    h = rng.random(n) + 0.01
    acc = rng.integers(-50, 51, (dim, n)).astype(float)
    acc[:, n // 3] = 0.0
    if n > 100:
        h[5], h[6], acc[0, 7] = np.nan, -1.0, np.inf
        h[7], acc[0, 8] = np.inf, np.nan
    h[n - 1], acc[:, n - 1] = 1e-3, 7.0  # the least, in the last place
    for hvs in (1e9, 1e-9):
        t = [torch.from_numpy(x.copy()).cuda() for x in (h, *acc, np.array([hvs]))]
        out = torch.zeros(1, dtype=torch.float64, device="cuda")
        p = [x.data_ptr() for x in t]
        rc = fn(dim, n, p[0], p[1], p[2] if dim > 1 else None, p[3] if dim > 2 else None, p[-1], 0.3, 0.125, out.data_ptr(),
                torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert rc == 0 and out.item() == _expected(h, acc, hvs, 0.3, 0.125)
