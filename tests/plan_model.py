"""The library's build plan and the row words of its count pass on the CPU (tests/plan_model.cpp,
built here with g++ from dynamis_amd/csrc/dg_plan.hpp)."""
import ctypes
import functools
import os
import subprocess
import tempfile
from types import SimpleNamespace

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(maxsize=None)
def _lib():
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "libplan_model.so")
        r = subprocess.run(["g++", "-std=c++17", "-O2", "-shared", "-fPIC",
                            os.path.join(HERE, "plan_model.cpp"), "-o", so], capture_output=True, text=True)
        assert r.returncode == 0, r.stderr
        lib = ctypes.CDLL(so)  # (stays mapped when the file is gone)
    lib.count_words.restype = ctypes.c_int64
    return lib


def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def _cell(cell, pbc):
    return np.ascontiguousarray(cell, np.float64).reshape(9), np.ascontiguousarray(pbc, np.uint8)


def plan(cell, pbc, radius, n, targets=None, f64=False):
    """The plan's numbers for n atoms (targets: how many explicit ones)."""
    c, b = _cell(cell, pbc)
    out = np.zeros(23, np.int64)
    bad = _lib().plan_numbers(_ptr(c), _ptr(b), ctypes.c_double(radius), ctypes.c_int64(n),
                              ctypes.c_int64(-1 if targets is None else targets), int(f64), _ptr(out))
    assert bad == 0
    v = [int(x) for x in out]
    return SimpleNamespace(nb=v[0:3], P=v[3:6], T=v[6:9], ntl=v[9:12], R=v[12:15], Kw=v[15], nrow=v[16],
                           mapcap=v[17], ws_bytes=v[18], all_pairs=bool(v[19]),
                           least_bytes=v[20], o_nw=v[21], npools=v[22])


def row_words(pos, cell, pbc, radius, f64=False):
    """(row words of every atom as a target, region-map entries that each pool is asked for first)."""
    c, b = _cell(cell, pbc)
    p = np.ascontiguousarray(pos, np.float64)
    words = np.zeros(len(p), np.int32)
    pools = np.zeros(64, np.int64)
    entries = int(_lib().count_words(_ptr(c), _ptr(b), ctypes.c_double(radius), ctypes.c_int64(len(p)), _ptr(p),
                                     int(f64), _ptr(words), _ptr(pools)))
    assert entries == pools.sum()
    return words, pools
