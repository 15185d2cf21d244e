"""csrc/m2l_plan.hpp through ctypes (a small library compiled by g++ on first use)."""
import ctypes
import functools
import os
import subprocess
import tempfile

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(maxsize=None)
def lib():
    tmp = tempfile.TemporaryDirectory(prefix="m2l_plan")
    out = os.path.join(tmp.name, "plan.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-shared", "-fPIC",
                    os.path.join(HERE, "plan.cpp"), "-o", out], check=True)
    L = ctypes.CDLL(out)
    tmp.cleanup()  # the loaded library stays
    L.plan_nowhere.restype = ctypes.c_uint32
    L.plan_two_tiles.argtypes = [ctypes.c_int64]
    L.plan_room.restype = ctypes.c_uint64
    L.plan_room.argtypes = [ctypes.c_uint64] * 4
    L.plan_cut.restype = ctypes.c_uint64
    L.plan_cut.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int64, ctypes.c_uint64,
                           ctypes.c_uint64, ctypes.c_void_p, ctypes.c_void_p]
    return L


def two_tiles(ncell):
    """Whether a workgroup takes two column tiles (32 cells)."""
    return bool(lib().plan_two_tiles(int(ncell)))


def rows(rank):
    """(offset index, place, largest place with signs) of every row and the bytes before each row block."""
    rank = np.ascontiguousarray(rank, np.int32)
    tau, off, last = (np.zeros(16 * 256, np.uint32) for _ in range(3))
    rboff = np.zeros(257, np.int32)
    nrb = lib().plan_rows(*(a.ctypes.data_as(ctypes.c_void_p) for a in (rank, tau, off, last, rboff)))
    n = 16 * nrb
    return tau[:n], off[:n], last[:n], rboff[: nrb + 1]


def cut(rboff, step, max_part, ncell, acc, room):
    """(first row blocks of the parts and the end, bytes of C)"""
    rboff = np.ascontiguousarray(rboff, np.int32)
    out = np.zeros(len(rboff) + 1, np.int32)
    parts = ctypes.c_int()
    size = lib().plan_cut(rboff.ctypes.data, len(rboff) - 1, step, max_part, ncell, acc, room, out.ctypes.data,
                          ctypes.addressof(parts))
    return out[: parts.value + 1], size
