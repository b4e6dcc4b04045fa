"""The grouped M2L (k_m2l_grp) against the M2L one pair at a time (k_m2l,
FMM3D_M2L_ROTATION=pairs) at the orders of iprec -2 .. 4 (2, 5, 9, 14, 26, 39
and 51), hence at every launch shape they take: eight, four and one group at a
time, one and two work items per thread, four, two and one members per group.
(Order 64 of iprec 5 has more work items than a workgroup takes and runs one
pair at a time itself.)  The two sum the same terms in another order: a local coefficient
is a sum of at most 189 translations of about p products, so FP64 results agree
to 1e-12 and FP32 ones to 1e-5 of their norm.  The switch is read once per
process, so the pairs run in a child."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
IPRECS = [-2, -1, 0, 1, 2, 3, 4]
CHILD = r"""
import sys
sys.path.insert(0, HERE)
import numpy as np
import test_gpu_m2l_groups as t
np.savez(OUT, **{"%d_%s_%d" % k: v for k, v in t.results().items()})
"""


def results():
    import fmmlib3d_amd as F
    from fmm_inputs import LEAF_SIZE, tree_work
    rng = np.random.default_rng(31)
    out = {}
    for iprec in IPRECS:
        for dist in ("cube", "shell"):
            # levels 2 and 3 filled, at the highest orders level 2 (a shell has
            # partial classes: groups of one and two members)
            n = (130 if iprec < 3 else 16) * LEAF_SIZE[iprec] + 1
            x = rng.random((n, 3))
            if dist == "shell":
                x = (x - 0.5) / np.linalg.norm(x - 0.5, axis=1, keepdims=True)
            assert tree_work(iprec, x)["list2"] > 2000
            q = rng.standard_normal(n) + 1j * rng.standard_normal(n)
            for prec in (F.PREC_FP64, F.PREC_FP32):
                ier, pot = F.lfmm3dpartself(iprec, x, q, None, None, iffld=0, precision=prec)[:2]
                assert ier == 0
                out[(iprec, dist, prec)] = pot
    return out


def test_gpu_m2l_groups_match_pairs(tmp_path):
    import fmmlib3d_amd as F
    path = str(tmp_path / "pairs.npz")
    r = subprocess.run([sys.executable, "-c", "HERE = %r\nOUT = %r\n" % (HERE, path) + CHILD],
                       env=dict(os.environ, FMM3D_M2L_ROTATION="pairs", PYTHONPATH=os.path.dirname(HERE)),
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=110)
    assert r.returncode == 0, r.stdout[-2000:]
    with np.load(path) as want:
        for (iprec, dist, prec), pot in results().items():
            ref = want["%d_%s_%d" % (iprec, dist, prec)]
            err = np.linalg.norm(pot - ref) / np.linalg.norm(ref)
            assert err < (1e-12 if prec == F.PREC_FP64 else 1e-5), (iprec, dist, prec, err)
