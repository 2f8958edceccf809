"""A device with little memory left, for tests of what a call does then."""
import contextlib
import ctypes as C

import prism_amd as P


@contextlib.contextmanager
def full_device(leave):
    """Holds the device's memory but for `leave` bytes or up to 16 MB more; gives the bytes left."""
    rt = P.hip_lib().dll  # the HIP runtime's calls are found through the library that links it
    held = []

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert rt.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    try:
        for chunk in (8 << 30, 512 << 20, 16 << 20):
            while free() >= chunk + leave:
                p = C.c_void_p()
                assert rt.hipMalloc(C.byref(p), C.c_size_t(chunk)) == 0
                held.append(p)
        yield free()
    finally:
        for p in held:
            rt.hipFree(p)
