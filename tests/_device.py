"""Device memory as the HIP runtime that the library maps reports it."""
import ctypes

import golaypair_amd as g


def held_by(call):
    """(result of call(ctx), bytes of device memory that its new context holds after it)."""
    g.load_library()
    path = next(l.split()[-1] for l in open("/proc/self/maps") if "libamdhip64" in l)
    hip = ctypes.CDLL(path)

    def free():
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    ctx = g.Context(0)
    try:
        before = free()
        out = call(ctx)
        return out, before - free()
    finally:
        ctx.close()
