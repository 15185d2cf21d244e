"""Takes device memory, as another program on the card would."""
import contextlib
import ctypes

from scalfmm_amd import _abi


@contextlib.contextmanager
def all_but(left):
    """Holds the free device memory except about `left` bytes; 0: all that the
    runtime gives in pieces of 4 MiB, whatever it says is free (it keeps some of its own)."""
    hip = _abi.lib()  # the runtime that the engine is bound to
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    held = []

    def take(size):
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)):
            hip.hipGetLastError()
            return False
        held.append(p)
        return True

    try:
        for size in (4 << 30, 256 << 20, 16 << 20, 4 << 20):
            while True:
                if hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)):
                    raise RuntimeError("hipMemGetInfo")
                if (left and free.value < left + size) or not take(size):
                    break
        yield free.value
    finally:
        for p in held:
            hip.hipFree(p)
