"""Device arrays and streams for the GPU tests through the HIP runtime that the
library itself links (torch would bring a second one into the process)."""
import ctypes
import os

import numpy as np


def runtime():
    rt = ctypes.CDLL(os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib", "libamdhip64.so"))
    rt.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
    rt.hipFree.argtypes = [ctypes.c_void_p]
    rt.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    rt.hipStreamCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    rt.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    rt.hipMemGetInfo.argtypes = [ctypes.POINTER(ctypes.c_size_t), ctypes.POINTER(ctypes.c_size_t)]
    return rt


class DeviceArrays:
    """Arrays freed and streams destroyed together at the end of a `with`."""

    def __init__(self):
        self.rt, self.bufs, self.streams = runtime(), [], []

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        assert self.rt.hipDeviceSynchronize() == 0
        for p in self.bufs:
            self.rt.hipFree(p)
        for s in self.streams:
            self.rt.hipStreamDestroy(s)

    def stream(self):
        s = ctypes.c_void_p()
        assert self.rt.hipStreamCreate(ctypes.byref(s)) == 0
        self.streams.append(s)
        return s

    def put(self, a):
        """A device copy of the array `a`."""
        a = np.ascontiguousarray(a)
        p = ctypes.c_void_p()
        assert self.rt.hipMalloc(ctypes.byref(p), max(a.nbytes, 8)) == 0
        self.bufs.append(p)
        assert self.rt.hipMemcpy(p, a.ctypes.data_as(ctypes.c_void_p), a.nbytes, 1) == 0
        return p

    def get(self, p, shape, dtype=np.complex128):
        """The device array at `p` as a host array."""
        a = np.zeros(shape, dtype)
        assert self.rt.hipMemcpy(a.ctypes.data_as(ctypes.c_void_p), p, a.nbytes, 2) == 0
        return a
