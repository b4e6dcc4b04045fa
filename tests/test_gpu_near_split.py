"""The near field's work split (GPU, against the oracle's sums over all pairs):
the four waves of a workgroup share 64 evaluation points and take quarters of
every source box; sources and targets go into one launch where both want the
same outputs.  Calls whose points fit one leaf are the near field alone; sizes
sit at the edges of the quarters (fewer sources than waves, one more than a
multiple), at those of the FP32 runs of 32 sources (quarters of 31 to 33 and 63
to 65), at multiples of 64 points and at item counts that are no multiple of
four.

A sum of n terms in another order moves by about sqrt(n) eps of its terms'
norm; 1e-12 leaves two digits for the cancellation of random signs at these
sizes.  The FP32 near field rounds each pair to 6e-8 except the closest, which
run in FP64: 1e-6, a digit for the cancellation."""
import numpy as np
import pytest

import fmmlib3d_amd as F
import oracle_bindings as ob
from fmm_inputs import points, rel, strengths, tree_work

pytestmark = pytest.mark.gpu


def _compare(got, want, flags, tol):
    for g, w, on in zip(got, want, flags):
        if not on:
            assert g is None
        elif np.linalg.norm(w) > 0:
            assert rel(g, w) < tol
        else:
            assert np.linalg.norm(g) == 0


def _check(rng, ns, nt, chg, dip, flags=(1, 1, 1, 1), iprec=6, prec=F.PREC_FP64, tol=1e-12):
    src = points(rng, ns, "cube")
    trg = points(rng, nt, "cube")
    q, ds, dv = strengths(rng, ns, chg, dip)
    ier, *got = F.lfmm3dparttarg(iprec, src, q, ds, dv, trg, *flags, precision=prec)
    assert ier == 0 and F.last_precision() == prec
    _compare(got, ob.orc_l3dpartdirect(src, q, ds, dv, trg), flags, tol)


@pytest.mark.parametrize("ns", [1, 2, 3, 4, 5, 8, 9, 63, 64, 65, 127, 128, 129, 513])
@pytest.mark.parametrize("chg,dip", [(True, False), (False, True), (True, True)])
def test_gpu_near_split_small(ns, chg, dip):
    _check(np.random.default_rng(ns), ns, 70, chg, dip)


@pytest.mark.parametrize("ns", [1, 3, 5, 124, 125, 128, 129, 131, 133, 252, 257, 260, 399])
@pytest.mark.parametrize("chg,dip", [(True, False), (True, True)])
def test_gpu_near_split_fp32_runs(ns, chg, dip):
    """One leaf at iprec 2 (leaf size 400)."""
    _check(np.random.default_rng(ns), ns, 70, chg, dip, iprec=2, prec=F.PREC_MIXED, tol=1e-6)


FLAGS = [(1, 0, 1, 1), (1, 1, 1, 0), (0, 1, 1, 1), (1, 1, 0, 0), (0, 0, 1, 1), (1, 0, 1, 0), (0, 1, 0, 1)]


@pytest.mark.parametrize("flags", FLAGS)
@pytest.mark.parametrize("ns,nt", [(300, 200), (65, 64), (64, 1)])
def test_gpu_near_split_flags(flags, ns, nt):
    """One launch and two, with one to five work items of a kind."""
    _check(np.random.default_rng(5), ns, nt, True, True, flags)


@pytest.mark.parametrize("flags", FLAGS + [(1, 1, 1, 1)])
def test_gpu_near_split_leaves(flags):
    """Many leaves of up to 80 points, against the oracle's FMM, which truncates
    alike (1e-11: P2M to L2P besides)."""
    rng = np.random.default_rng(6)
    src, trg = points(rng, 4001, "shell"), points(rng, 2003, "cube")
    q, ds, dv = strengths(rng, 4001, True, True)
    assert tree_work(0, src, trg)["p2m"] > 50
    ier, *got = F.lfmm3dparttarg(0, src, q, ds, dv, trg, *flags)
    assert ier == 0
    want = ob.orc_lfmm3dparttarg(0, src, q, ds, dv, trg)
    _compare(got, want[1:], flags, 1e-11)
