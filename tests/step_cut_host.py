"""The decode step's plan and cut (``csrc/step_plan.h``, ``csrc/step_cut.h``) built for the host."""
import ctypes
import pathlib
import subprocess
import tempfile
import types

import numpy as np

HERE = pathlib.Path(__file__).resolve().parent
CUS = 256
_lib = None


def lib():
    global _lib
    if _lib is None:
        with tempfile.TemporaryDirectory() as d:
            so = pathlib.Path(d) / "step_cut_host.so"
            subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-U_FORTIFY_SOURCE", "-o", str(so),
                            str(HERE / "step_cut_host.cpp")], check=True)
            _lib = ctypes.CDLL(str(so))
        _lib.host_segments.argtypes = [ctypes.c_void_p] + [ctypes.c_int] * 6 + [ctypes.c_void_p, ctypes.c_int]
    return _lib


def waves():
    """Waves per workgroup at most."""
    return lib().host_waves()


def plan(batch, nvh, max_blocks, splits, *, block_size=16, whole_lines=True, have_parts=True):
    """``step_plan`` on 256 CUs; ``nvh``: head parts of a sequence."""
    out = (ctypes.c_int * 6)()
    lib().host_step_plan(CUS * waves(), nvh, batch, max_blocks, block_size, splits, int(whole_lines),
                         int(have_parts and splits > 1), out)
    return types.SimpleNamespace(vw=out[0], sw=out[1], nx=out[2], per_seq=out[3], whole=bool(out[4]),
                                 rotates=bool(out[5]))


def segments(lens, splits, p, x):
    """(sequence, first tile, end tile, part, parts) of workgroup ``x`` of plan ``p``."""
    if p.whole:
        tiles = (max(int(lens[x]), 0) + 15) >> 4
        return [(x, 0, tiles, 0, 1)] if tiles else []
    lens = np.ascontiguousarray(lens, np.int32)
    room = len(lens) + 1
    out = np.zeros((room, 5), np.int32)
    n = lib().host_segments(lens.ctypes.data, len(lens), splits, p.sw, p.per_seq, p.nx, x, out.ctypes.data, room)
    assert n >= 0, (n, x)
    return [tuple(int(v) for v in row) for row in out[:n]]


def run_of(tiles, n, i):
    """[first, end) of run ``i`` of ``n``."""
    first, count = ctypes.c_int(), ctypes.c_int()
    lib().host_run(int(tiles), int(n), int(i), ctypes.byref(first), ctypes.byref(count))
    return first.value, first.value + count.value
