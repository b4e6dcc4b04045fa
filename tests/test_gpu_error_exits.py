"""A call that fails after it has queued work must not reach into the next one,
which may come on another stream: refused Helmholtz orders between good calls
(tables, pinned buffers and cached operators are the context's), with the tree
built on the device and on the host, and a fixed workspace that runs out half
way through a call.  The good calls are compared with the oracle's FMM, which
truncates alike (1e-10, as elsewhere), and repeated ones bitwise."""
import ctypes

import numpy as np
import pytest

import fmmlib3d_amd as F
import oracle_bindings as ob
from fmm_inputs import points, rel, strengths
from hip_arrays import DeviceArrays

pytestmark = pytest.mark.gpu


def _dev_call(D, fn, head, x, q, stream):
    """One self-interaction call with charges on `stream`: (ier, pot, fld)."""
    n = len(x)
    tx, tq, pot, fld = D.put(x), D.put(q), D.put(np.zeros(n, complex)), D.put(np.zeros((n, 3), complex))
    ier = fn(*head, n, tx, 1, tq, 0, None, None, 1, pot, 1, fld, 0, None, 0, None, 0, None, stream)
    return ier, D.get(pot, n), D.get(fld, (n, 3))


@pytest.mark.parametrize("tree", ["device", "host"])
def test_gpu_refused_order_between_calls(tree, monkeypatch):
    monkeypatch.setenv("FMM3D_TREE", tree)
    lib = F.load()
    x = points(np.random.default_rng(1), 3000, "clusters")
    q, _, _ = strengths(np.random.default_rng(2), 3000)
    first = {}
    with DeviceArrays() as D:
        streams = [D.stream(), D.stream()]
        # the order at zk = 250 on this box does not fit the kernels' LDS; at 500
        # it is beyond what the tables are made for
        for k, zk in enumerate([6.0, 250.0, 9.0, 500.0, 6.0, 250.0, 6.0, 9.0]):
            z = np.array([zk, 0.0])
            head = (0, 2, z.ctypes.data_as(ctypes.c_void_p))
            ier, pot, fld = _dev_call(D, lib.fmm3d_hfmm3dparttarg_dev, head, x, q, streams[k % 2])
            assert ier == (16 if zk > 100 else 0), (zk, ier)
            if ier:
                continue
            if zk not in first:
                first[zk] = (pot, fld)
                want = ob.orc_hfmm3dparttarg(2, zk, x, q)
                assert rel(pot, want[1]) < 1e-10 and rel(fld, want[2]) < 1e-10
            assert np.array_equal(pot, first[zk][0]) and np.array_equal(fld, first[zk][1])


def test_gpu_workspace_runs_out_between_calls():
    lib = F.load()
    rng = np.random.default_rng(3)
    big = points(rng, 400000, "clusters")
    qb, _, _ = strengths(rng, 400000)
    x = points(rng, 20000, "clusters")
    q, _, _ = strengths(rng, 20000)
    with DeviceArrays() as D:
        streams = [D.stream(), D.stream()]
        want = _dev_call(D, lib.fmm3d_lfmm3dparttarg_dev, (0, 1), x, q, streams[0])
        assert want[0] == 0
        for k in range(4):
            # its tree and tables fit the region, its expansions or packs do not
            assert _dev_call(D, lib.fmm3d_lfmm3dparttarg_dev_noalloc, (0, 2), big, qb, streams[k % 2])[0] == 256
            got = _dev_call(D, lib.fmm3d_lfmm3dparttarg_dev_noalloc, (0, 1), x, q, streams[1 - k % 2])
            assert got[0] == 0
            assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])
