"""The Helmholtz operators computed on the device (GPU, against the oracle's
FMM): wavenumbers, root boxes, depths and tolerances in turn on one context, so
that each call replaces another part of the tables (operators alone, then also
the geometry of another order, then the integrals of a larger one) or none; a
tree of two levels has M2L operators only, one of a single leaf none.  Bar as
for the other comparisons with the oracle's FMM, which truncates alike."""
import numpy as np
import pytest

import fmmlib3d_amd as F
import oracle_bindings as ob
from fmm_inputs import points, rel, strengths

pytestmark = pytest.mark.gpu

# (zk, iprec, sources, scale of the box)
CALLS = [(6.0, 2, 2500, 1.0), (6.0, 2, 2500, 1.3), (6.0 + 0.4j, 2, 2500, 1.3), (6.0, 2, 2500, 1.0), (6.0, 3, 3000, 1.0),
         (14.0, 0, 2500, 1.0), (14.0, 0, 20, 1.0), (0.5, 1, 400, 1.0), (25.0, 2, 2500, 1.0), (6.0, 2, 2500, 1.0)]


def test_gpu_helm_tables_in_turn():
    first = {}
    for zk, iprec, ns, scale in CALLS:
        rng = np.random.default_rng(ns)
        src = scale * points(rng, ns, "clusters" if ns == 2500 else "cube")
        q, ds, dv = strengths(rng, ns, True, True)
        trg = scale * points(rng, 300, "cube")
        got = F.hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
        want = ob.orc_hfmm3dparttarg(iprec, zk, src, q, ds, dv, trg)
        assert got[0] == 0 and want[0] == 0
        for g, w in zip(got[1:], want[1:]):
            assert rel(g, w) < 1e-10
        key = (zk, iprec, ns, scale)
        if key in first:  # the tables of a call repeated later are the same
            for g, w in zip(got[1:], first[key][1:]):
                assert np.array_equal(g, w)
        first[key] = got
