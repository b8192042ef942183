"""The HIP runtime that the library has loaded, for tests that need device memory of their own (a
second runtime beside it, such as torch's when it is imported later, finds no GPU)."""
import ctypes as C

import numpy as np


def _hip():
    hip = C.CDLL("libamdhip64.so.7")  # by its soname: the one in the process
    hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
    hip.hipFree.argtypes = [C.c_void_p]
    hip.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
    hip.hipMemGetInfo.argtypes = [C.POINTER(C.c_size_t), C.POINTER(C.c_size_t)]
    return hip


def memory_used():
    """Bytes of the current device in use."""
    hip, free, total = _hip(), C.c_size_t(), C.c_size_t()
    assert hip.hipDeviceSynchronize() == 0
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return total.value - free.value


class DeviceArray:
    """A device copy of a numpy array."""

    def __init__(self, a):
        self.hip, self.host, self.ptr = _hip(), np.ascontiguousarray(a), C.c_void_p()
        assert self.hip.hipMalloc(C.byref(self.ptr), self.host.nbytes) == 0
        assert self.hip.hipMemcpy(self.ptr, self.host.ctypes.data, self.host.nbytes, 1) == 0

    def get(self):
        out = np.empty_like(self.host)
        assert self.hip.hipMemcpy(out.ctypes.data, self.ptr, out.nbytes, 2) == 0
        return out

    def close(self):
        self.hip.hipFree(self.ptr)
