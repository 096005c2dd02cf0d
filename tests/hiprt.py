"""The HIP runtime that libhegjoin.so has loaded, through ctypes (torch brings a
second one, which finds no device after the first has)."""
import ctypes as C

import numpy as np


def runtime():
    import hegjoin_amd  # noqa: F401 (loads the runtime)
    rt = C.CDLL("libamdhip64.so.7")
    rt.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    rt.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    rt.hipFree.argtypes = rt.hipHostFree.argtypes = [C.c_void_p]
    rt.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    rt.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    return rt


def free_bytes(rt):
    free, total = C.c_size_t(), C.c_size_t()
    assert rt.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


class Buf:
    """Device memory, or host memory that the runtime pinned."""

    def __init__(self, rt, dtype, count, pinned=False):
        self.rt, self.dtype, self.count, self.pinned = rt, np.dtype(dtype), count, pinned
        self.nbytes, p = self.dtype.itemsize * count, C.c_void_p()
        if pinned:
            assert rt.hipHostMalloc(C.byref(p), max(self.nbytes, 16), 0) == 0
        else:
            assert rt.hipMalloc(C.byref(p), max(self.nbytes, 16)) == 0
        self.p = p.value

    def get(self):
        out = np.empty(self.count, self.dtype)
        if self.count:
            assert self.rt.hipMemcpy(out.ctypes.data, self.p, self.nbytes, 0 if self.pinned else 2) == 0
        return out

    def free(self):
        (self.rt.hipHostFree if self.pinned else self.rt.hipFree)(self.p)
