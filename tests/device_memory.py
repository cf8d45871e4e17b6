"""Device memory through the HIP runtime that the engine loaded (a second
runtime in the process would not see the device)."""
import ctypes

from cafe5_amd import native

MB = 1 << 20


def _rt():
    return native.load_library()   # (its dependencies' symbols too)


def free_bytes() -> int:
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _rt().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


class Filled:
    """Holds all device memory but about `left` bytes."""

    def __init__(self, left: int):
        lib = _rt()
        lib.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
        lib.hipFree.argtypes = [ctypes.c_void_p]
        self.blocks = []
        for size in (64 << 30, 8 << 30, 1 << 30, 16 * MB):
            while True:
                p = ctypes.c_void_p()
                if lib.hipMalloc(ctypes.byref(p), size) != 0:
                    lib.hipGetLastError()
                    break
                self.blocks.append(p)
        n = left // (16 * MB)
        assert len(self.blocks) > n
        for _ in range(n):
            lib.hipFree(self.blocks.pop())

    def release(self):
        while self.blocks:
            _rt().hipFree(self.blocks.pop())
