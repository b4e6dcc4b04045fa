"""The Helmholtz operators computed on the device (GPU, against the oracle's
FMM).

In turn: wavenumbers, root boxes, depths and tolerances one after the other on
one context, so that each call replaces another part of the tables (operators
alone, then also the geometry of another order, then the integrals of a larger
one) or none; a tree of two levels has M2L operators only, one of a single leaf
none.  Bar as for the other comparisons with the oracle's FMM, which truncates
alike.

By order: the grouped M2L with complex shift tables (k_hm2l_grp) at each launch
shape, eight, four and one group at a time, one and two work items per thread,
and the order beyond it that runs one pair at a time.  The terms of a shift
cancel the more the larger the box is in wavelengths; above order 42 (150 and
180 radians across) ten times the bar."""
import ctypes

import numpy as np
import pytest

import fmmlib3d_amd as F
import oracle_bindings as ob
from fmm_inputs import IPREC_EPS, LEAF_SIZE, points, rel, strengths, tree_work

pytestmark = pytest.mark.gpu

# (zk, iprec, sources, their distribution, scale of the box, levels of the tree)
CALLS = [(6.0, 2, 2500, "clusters", 1.0, 3), (6.0, 2, 2500, "clusters", 1.3, 3),
         (6.0 + 0.4j, 2, 2500, "clusters", 1.3, 3), (6.0, 2, 2500, "clusters", 1.0, 3),
         (6.0, 3, 9000, "clusters", 1.0, 4), (14.0, 0, 2500, "clusters", 1.0, 5), (14.0, 2, 20, "cube", 1.0, 0),
         (0.5, 1, 1600, "cube", 1.0, 2), (25.0, 2, 2500, "clusters", 1.0, 3), (6.0, 2, 2500, "clusters", 1.0, 3)]


def test_gpu_helm_tables_in_turn():
    first = {}
    for call in CALLS:
        zk, iprec, ns, dist, scale, levels = call
        rng = np.random.default_rng(ns)
        src = scale * points(rng, ns, dist)
        q, ds, dv = strengths(rng, ns, True, True)
        trg = scale * points(rng, 300, "cube")
        work = tree_work(iprec, src, trg)
        assert work["levels"] == levels and (work["list2"] > 0) == (levels >= 2)
        got = F.hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
        want = ob.orc_hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
        assert got[0] == 0 and want[0] == 0
        for g, w in zip(got[1:], want[1:]):
            assert rel(g, w) < 1e-10
        if call in first:  # the tables of a call repeated later are the same
            for g, w in zip(got[1:], first[call][1:]):
                assert np.array_equal(g, w)
        first[call] = got


def order(size, zk, eps):
    """The expansion order of a box (src/h3dterms.f), from the oracle."""
    o = ob.oracle()
    o.orc_h3dterms.argtypes = [ctypes.c_double, ob.ZC, ctypes.c_double, ctypes.c_void_p]
    o.orc_h3dterms.restype = ctypes.c_int
    return o.orc_h3dterms(size, ob.zc(zk), eps, ctypes.byref(ctypes.c_int(0)))


# (zk, iprec, least and largest order of the launch shape)
@pytest.mark.parametrize("zk,iprec,lo,hi", [(6.0, 1, 1, 13), (30.0, 1, 14, 19), (6.0, 2, 20, 29), (100.0, 2, 30, 42),
                                            (150.0, 2, 43, 61), (180.0, 2, 62, 62)])
def test_gpu_helm_m2l_orders(zk, iprec, lo, hi):
    rng = np.random.default_rng(int(zk))
    ns, nt = 16 * LEAF_SIZE[iprec], 500
    src, trg = rng.random((ns, 3)), rng.random((nt, 3))
    src[0], src[1] = 0.0, 1.0                    # the root box is the unit cube
    assert lo <= order(0.25, zk, IPREC_EPS[iprec]) <= hi
    assert tree_work(iprec, src, trg)["list2"] > 2000
    q, ds, dv = strengths(rng, ns, True, True)
    got = F.hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
    want = ob.orc_hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
    assert got[0] == 0 and want[0] == 0
    for g, w in zip(got[1:], want[1:]):
        assert rel(g, w) < (1e-10 if hi <= 42 else 1e-9)
