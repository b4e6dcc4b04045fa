"""Calls near the size that the fixed workspace of
fmm3d_lfmm3dparttarg_dev_noalloc holds: what it took it keeps taking (sizes
within 2,000 points of the limit from before the packed expansions, the
strengths and the tables grew), with the results of fmm3d_lfmm3dparttarg_dev
bit for bit."""
import numpy as np
import pytest

import fmmlib3d_amd as F
from fmm_inputs import points
from hip_arrays import DeviceArrays

pytestmark = pytest.mark.gpu

# (precision mode, iprec, distribution, sources = targets)
LIMITS = [(0, 2, "clusters", 65500), (0, 0, "cube", 270000), (0, 2, "plummer", 87000), (0, 1, "clusters", 106500),
          (0, 3, "cube", 80000), (0, -2, "cube", 458000), (2, 1, "cube", 486000), (2, -2, "cube", 498000),
          (2, 1, "clusters", 161500)]


@pytest.mark.parametrize("prec,iprec,dist,n", LIMITS)
def test_gpu_workspace_limit(prec, iprec, dist, n):
    rng = np.random.default_rng(n)
    x, y = points(rng, n, dist), points(rng, n, dist)
    q, ds = (rng.standard_normal(n) + 1j * rng.standard_normal(n) for _ in range(2))
    dv = rng.standard_normal((n, 3))
    shapes = [(n,), (n, 3), (n,), (n, 3)]
    with DeviceArrays() as D:
        x, q, ds, dv, y = (D.put(a) for a in (x, q, ds, dv, y))
        res = []
        for name in ("fmm3d_lfmm3dparttarg_dev_noalloc", "fmm3d_lfmm3dparttarg_dev"):
            p, f, pt, ft = (D.put(np.zeros(s, complex)) for s in shapes)
            assert getattr(F.load(), name)(prec, iprec, n, x, 1, q, 1, ds, dv, 1, p, 1, f, n, y, 1, pt, 1, ft, None) == 0
            res.append([D.get(a, s) for a, s in zip((p, f, pt, ft), shapes)])
    assert all(np.array_equal(a, b) for a, b in zip(*res))
