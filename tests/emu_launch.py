"""The emulation's last launch: its mode bits and schedule."""
import ctypes

# mode bits (optifax_amd/csrc/ofx_backend.h)
BARRIER, RK23, SIZED, WAVE, FIXED = 1, 2, 4, 0x70, 0x1f00


def last_launch(ctx):
    """(mode, [(grid size, cluster index) of every instance in launch order])."""
    n, c, count = (ctypes.c_int * 1024)(), (ctypes.c_int * 1024)(), ctypes.c_int()
    mode = ctx.lib.ofx_emu_last_launch(1024, n, c, ctypes.byref(count))
    assert 0 <= mode and count.value <= 1024
    return mode, [(n[i], c[i]) for i in range(count.value)]


def kernel(mode):
    """Which kernel a mode names."""
    if mode & (WAVE | FIXED):
        return "wave rk23" if mode & RK23 else "wave"
    if mode & SIZED:
        return "sized"
    return ("rk23 " if mode & RK23 else "general ") + ("barrier" if mode & BARRIER else "tags")
