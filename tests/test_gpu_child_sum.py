"""M2M and L2L by child: trees whose level-2 boxes have one to eight children,
Laplace and Helmholtz, against the direct sum at sampled points.  The calls ask
for 0.5e-9 of the potential (iprec 3); 1e-8 leaves room for the sample."""
import numpy as np
import pytest

from fmm_inputs import tree_work

pytestmark = pytest.mark.gpu


def child_points(children):
    """900 points in each of the 64 boxes of level 2, which then split (leaf size
    800), in `children` of its octants; the corners of the root cube besides."""
    rng = np.random.default_rng(17 + children)
    cell = np.stack(np.meshgrid(*[np.arange(4)] * 3, indexing="ij"), -1).reshape(-1, 3)
    cell = np.repeat(cell, 900, axis=0)
    octant = (np.tile(np.arange(900), 64) % children * 3 + 1) % 8
    sub = np.stack([octant & 1, octant >> 1 & 1, octant >> 2 & 1], axis=1)
    x = (cell + 0.5 * (sub + rng.random(cell.shape))) / 4.0
    return np.concatenate([x, [[0.0, 0.0, 0.0], [1.0, 1.0, 1.0]]])


@pytest.mark.parametrize("zk", [0.0, 4.0])
@pytest.mark.parametrize("children", [1, 2, 3, 5, 7, 8])
def test_gpu_child_sum(children, zk):
    import fmmlib3d_amd as F
    x = child_points(children)
    n = len(x)
    kids = tree_work(3, x)["children_level2"]
    assert len(kids) == 64 and (kids == children).sum() >= 62   # (the corners may add an octant to two)
    rng = np.random.default_rng(children)
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
