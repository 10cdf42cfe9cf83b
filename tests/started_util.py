"""What a launch starts, as the library would enqueue it (no device is needed; 256 CUs are taken where there is none)."""
import ctypes

from orinfer_amd import lib

RUNS, BIG, MID_4, MID_2 = 163840, 133120, 131072, 65536  # dynamic LDS by which the kernels are told: channel runs, 256 x 256 tiles, 128 x 128 tiles of four and two stages


def started(kernel, rows=0):
    """(workgroups, threads, dynamic LDS bytes) of every kernel that a launch of `rows` rows enqueues, in order."""
    call = lib.library().orx_started_kernels
    call.argtypes = [ctypes.c_void_p, ctypes.c_int32, ctypes.c_void_p, ctypes.c_int32, ctypes.POINTER(ctypes.c_int32)]
    found, count = (ctypes.c_uint32 * 3 * 64)(), ctypes.c_int32()
    code = call(kernel._handle, rows, found, 64, ctypes.byref(count))
    if code != lib.ORX_OK:
        raise lib.OrxError(code, lib.last_error())
    return [tuple(found[i]) for i in range(count.value)]


def reported(kernel, rows=0):
    """The same of the kernel that orx_geometry describes."""
    grid, block, shared = kernel.geometry(rows)
    return grid[0], block[0] * block[1] * block[2], shared
