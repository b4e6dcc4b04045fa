"""P2M, P2L, M2P and L2P at every order they branch on (GPU, against the
oracle's FMM, which truncates alike): iprec -2 .. 4 are the orders 2, 5, 9, 14,
26, 39 and 51, i.e. one, two and four source groups, one and two entries per
thread, one or several ranges of orders and, for charges at 26 and 39, the
matrix cores.  Clustered sources against spread targets put boxes in lists 3
and 4 at every order; the box sizes leave partial tiles and batches.  The two sum the same
coefficients in another order; errors of 1e-15 per operation grow with the
condition of the recurrences (a factor 2 to 3 per ten degrees) and of the sums
over random signs: 1e-11 at orders up to 39, 1e-10 at 51."""
import numpy as np
import pytest

import fmmlib3d_amd as F
import oracle_bindings as ob
from fmm_inputs import LEAF_SIZE, points, rel, strengths, tree_work

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("iprec", [-2, -1, 0, 1, 2, 3, 4])
@pytest.mark.parametrize("chg,dip", [(True, False), (False, True), (True, True)])
def test_gpu_form_eval_orders(iprec, chg, dip):
    rng = np.random.default_rng(100 + iprec)
    ns, nt = max(4000, 12 * LEAF_SIZE[iprec]), max(1500, 2 * LEAF_SIZE[iprec])
    src = np.concatenate([points(rng, ns - 701, "clusters"), points(rng, 701, "cube")])
    trg = points(rng, nt, "cube")
    q, ds, dv = strengths(rng, ns, chg, dip)
    work = tree_work(iprec, src, trg)
    assert min(work["p2m"], work["list2"], work["list3"], work["list4"]) > 50
    got = F.lfmm3dparttarg(iprec, src, q, ds, dv, trg)
    want = ob.orc_lfmm3dparttarg(iprec, src, q, ds, dv, trg)
    assert got[0] == 0 and want[0] == 0
    for g, w in zip(got[1:], want[1:]):
        assert rel(g, w) < (1e-10 if iprec > 3 else 1e-11)


@pytest.mark.parametrize("ns", [1, 3, 4, 63, 64, 65, 129])
def test_gpu_form_small_boxes(ns):
    """One box of few sources: groups of four and batches of 64 not filled.  The
    targets make the tree: two levels, the sources inside one box of the second."""
    rng = np.random.default_rng(ns)
    src = 0.3 + 0.15 * rng.random((ns, 3))
    q, _, _ = strengths(rng, ns)
    for iprec, nt in ((1, 3000), (2, 8000)):
        trg = points(rng, nt, "cube")
        work = tree_work(iprec, src, trg)
        assert work["p2m"] == 1 and work["list2"] > 0
        got = F.lfmm3dparttarg(iprec, src, q, target=trg)
        want = ob.orc_lfmm3dparttarg(iprec, src, q, None, None, trg)
        assert got[0] == 0 and want[0] == 0
        for g, w in zip(got[1:], want[1:]):
            if np.linalg.norm(w) > 0:
                assert rel(g, w) < 1e-11
