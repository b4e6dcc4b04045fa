"""The near field's work split (GPU): the waves of a workgroup share 64
evaluation points and take parts of every source box, sixteen waves up to
1024 work items and four beyond.  iprec 6 makes one leaf of everything, so the
FMM is the near field alone and equals the direct sum; sizes sit at the edges
of the parts (fewer sources than waves, one more than a wave's points) and on
both sides of 1024 items.  A sum of n terms in another order moves by about
sqrt(n) eps of its terms' norm; 1e-12 leaves two digits for the cancellation
of random signs at these sizes."""
import numpy as np
import pytest

import fmmlib3d_amd as F
from fmm_inputs import points, rel, strengths

pytestmark = pytest.mark.gpu


def _check(rng, ns, nt, chg, dip, flags):
    src = points(rng, ns, "cube")
    trg = points(rng, nt, "cube")
    q, ds, dv = strengths(rng, ns, chg, dip)
    ier, *got = F.lfmm3dparttarg(6, src, q, ds, dv, trg, *flags)
    assert ier == 0
    want = F.l3dpartdirect(src, q, ds, dv, trg, *flags)
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        if g is not None and np.linalg.norm(w) > 0:
            assert rel(g, w) < 1e-12
        elif g is not None:
            assert np.linalg.norm(g) == 0


@pytest.mark.parametrize("ns", [1, 2, 3, 15, 16, 17, 31, 64, 65, 129, 511])
@pytest.mark.parametrize("chg,dip", [(True, False), (False, True), (True, True)])
def test_gpu_near_split_small(ns, chg, dip):
    _check(np.random.default_rng(ns), ns, 70, chg, dip, (1, 1, 1, 1))


@pytest.mark.parametrize("flags", [(1, 0, 1, 1), (1, 1, 1, 0), (0, 1, 1, 1), (1, 1, 0, 0), (0, 0, 1, 1), (1, 0, 1, 0)])
def test_gpu_near_split_flags(flags):
    _check(np.random.default_rng(5), 300, 200, True, True, flags)


@pytest.mark.parametrize("ns,nt", [(65472, 64), (65473, 64), (65537, 1)])
def test_gpu_near_split_either_side(ns, nt):
    _check(np.random.default_rng(ns), ns, nt, True, False, (1, 1, 1, 1))
