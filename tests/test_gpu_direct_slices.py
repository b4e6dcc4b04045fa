"""Direct sums at the edges of their split: one source per wave and fewer, one
slice and several, whole and ragged groups of 64 points.  Against the oracle's
sums, potential and field: a sum of at most 5,000 terms in FP64 differs by the
order of the terms, less than 5,000 x 2.2e-16 of the sum of their magnitudes:
1e-11 of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zk", [0.0, 3.0 + 0.2j])
@pytest.mark.parametrize("ns,nt", [(1, 1), (3, 64), (63, 65), (255, 1), (256, 63), (512, 130), (767, 64),
                                   (5000, 129), (129, 5000)])
def test_gpu_direct_sum_split(ns, nt, zk):
    import fmmlib3d_amd as F
    import oracle_bindings as ob
    rng = np.random.default_rng(1000 * ns + nt)
    x, y = rng.random((ns, 3)), rng.random((nt, 3)) + 0.01
    q, ds = (rng.standard_normal(ns) + 1j * rng.standard_normal(ns) for _ in range(2))
    dv = rng.standard_normal((ns, 3))
    if zk == 0.0:
        out, want = F.l3dpartdirect(x, q, ds, dv, y), ob.orc_l3dpartdirect(x, q, ds, dv, y)
    else:
        out, want = F.h3dpartdirect(zk, x, q, ds, dv, y), ob.orc_h3dpartdirect(zk, x, q, ds, dv, y)
    for name, got, ref in zip(("pot", "fld", "pottarg", "fldtarg"), out, want):
        assert got.shape == ref.shape
        err = np.linalg.norm(got - ref)
        assert err <= 1e-11 * np.linalg.norm(ref), (name, err)
