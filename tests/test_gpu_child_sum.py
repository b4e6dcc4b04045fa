"""M2M and L2L by child: trees whose parents have one to eight children, Laplace
and Helmholtz, against the direct sum at sampled points.  The calls ask for
0.5e-9 of the potential (iprec 3); 1e-8 leaves room for the sample."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zk", [0.0, 4.0])
@pytest.mark.parametrize("children", [1, 2, 3, 5, 7, 8])
def test_gpu_child_sum(children, zk):
    import fmmlib3d_amd as F
    rng = np.random.default_rng(17 + children)
    n = 20000
    cell = rng.integers(0, 4, (n, 3))            # level 2
    octant = (rng.integers(0, children, n) * 3 + 1) % 8 if children > 1 else np.zeros(n, int)
    octant = np.where(octant < 0, 0, octant)
    sub = np.stack([octant & 1, octant >> 1 & 1, octant >> 2 & 1], axis=1)
    x = (cell + 0.5 * (sub + rng.random((n, 3)))) / 4.0
    x[0], x[1] = 0.0, 1.0                        # the root cube
    q = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    if zk == 0.0:
        ier, pot, _ = F.lfmm3dpartself(3, x, q, iffld=0)
    else:
        ier, pot, _ = F.hfmm3dpartself(3, zk, x, q, iffld=0)
    assert ier == 0
    idx = rng.choice(n, 200, replace=False)
    r = np.linalg.norm(x[idx, None, :] - x[None, :, :], axis=2)
    r[np.arange(200), idx] = np.inf
    want = (np.exp(1j * zk * np.where(np.isinf(r), 0.0, r)) / r) @ q
    assert np.linalg.norm(pot[idx] - want) < 1e-8 * np.linalg.norm(want)
