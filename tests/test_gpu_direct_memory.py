"""Device memory of a direct sum: a few sources on many targets take no buffer
for sums of slices, since one slice is all there is.  In a child process, so
that no other call has grown the buffers before."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))

CHILD = r"""
import ctypes, sys
sys.path.insert(0, HERE)
import numpy as np
import fmmlib3d_amd as F
import hip_arrays
rt = hip_arrays.runtime()
def free():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert rt.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value
rng = np.random.default_rng(1)
x, q = rng.random((4, 3)), rng.standard_normal(4) + 0j
y = rng.random((3000000, 3))
call = (lambda z, y: F.l3dpartdirect(x, q, None, None, y, 0, 0, 1, 1)) if ZK == 0 else (
    lambda z, y: F.h3dpartdirect(ZK, x, q, None, None, y, 0, 0, 1, 1))
call(0, y[:10])
before = free()
pot = call(0, y)[2]
print("taken", before - free(), float(np.abs(pot).sum()))
"""


@pytest.mark.parametrize("zk", [0.0, 2.0])
def test_gpu_direct_memory(zk):
    r = subprocess.run([sys.executable, "-c", "HERE = %r\nZK = %r\n" % (HERE, zk) + CHILD],
                       env=dict(os.environ, PYTHONPATH=os.path.dirname(HERE)), stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=110)
    assert r.returncode == 0, r.stdout[-2000:]
    word, taken, total = r.stdout.split()[-3:]
    assert word == "taken" and float(total) > 0
    # bytes per target: order 4, positions in and sorted 24 + 32, potential and
    # field computed 16 + 48 and returned 16 + 48; buffers are taken an eighth
    # larger, and 32 MiB allow for their rounding
    assert int(taken) <= 1.125 * 188 * 3000000 + (32 << 20)
