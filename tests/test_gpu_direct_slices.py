"""Direct sums at the edges of their split: one source per wave and fewer, one
slice and several, whole and ragged groups of 64 points.  Against the sum in
numpy: a sum of at most 5,000 terms in FP64 differs by the order of the terms,
less than 5,000 x 2.2e-16 of the sum of their magnitudes: 1e-11 of the norm."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def reference(x, q, ds, dv, y, self_sum, zk):
    d = y[:, None, :] - x[None, :, :]
    r = np.sqrt((d * d).sum(-1))
    if self_sum:
        np.fill_diagonal(r, np.inf)
    e = np.exp(1j * zk * np.where(np.isinf(r), 0.0, r))
    g = (1 - 1j * zk * np.where(np.isinf(r), 0.0, r)) * e / r**3   # -grad(e^{ikr}/r) = g d
    pot = (e / r) @ q + (np.einsum("ijk,jk->ij", d, dv) * g) @ ds
    return pot


@pytest.mark.parametrize("zk", [0.0, 3.0 + 0.2j])
@pytest.mark.parametrize("ns,nt", [(1, 1), (3, 64), (63, 65), (255, 1), (256, 63), (512, 130), (767, 64),
                                   (5000, 129), (129, 5000)])
def test_gpu_direct_sum_split(ns, nt, zk):
    import fmmlib3d_amd as F
    rng = np.random.default_rng(1000 * ns + nt)
    x, y = rng.random((ns, 3)), rng.random((nt, 3)) + 0.01
    q, ds = (rng.standard_normal(ns) + 1j * rng.standard_normal(ns) for _ in range(2))
    dv = rng.standard_normal((ns, 3))
    if zk == 0.0:
        out = F.l3dpartdirect(x, q, ds, dv, y)
    else:
        out = F.h3dpartdirect(zk, x, q, ds, dv, y)
    for got, pts, own in ((out[0], x, True), (out[2], y, False)):
        want = reference(x, q, ds, dv, pts, own, zk)
        err = np.linalg.norm(got - want)
        assert err <= 1e-11 * np.linalg.norm(want), (own, err)
