"""Member segments (skg_seg.h, compiled for the host): whatever ids are missing, every member is found in its
own group and group 0's in none."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skid_amd", "csrc")


@pytest.fixture(scope="module")
def seg(tmp_path_factory):
    d = tmp_path_factory.mktemp("seg")
    src, so = d / "seg.cpp", d / "libseg.so"
    src.write_text('#define SKG_SEG_FN static inline\n#include "skg_seg.h"\n'
                   'extern "C" int start(const unsigned long long *k, int n, int g) { return group_start(k, n, g); }\n'
                   'extern "C" int at(const int *gs, const int *ge, int nG, int t) '
                   '{ return group_at(gs, ge, nG, t); }\n')
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(src)], check=True)
    lib = C.CDLL(str(so))
    lib.start.argtypes = [C.c_void_p, C.c_int, C.c_int]
    lib.at.argtypes = [C.c_void_p, C.c_void_p, C.c_int, C.c_int]
    return lib


@pytest.mark.parametrize("grp", [
    [0, 0, 0],                       # no group
    [1, 1, 2],                       # nobody outside
    [0, 1, 1, 3, 3, 0],              # an id missing between two groups
    [2, 2],                          # the first id missing
    [0, 5, 5, 5, 9, 0, 12, 12],      # several in a row
    [7],
])
def test_members_and_starts(seg, grp):
    grp = np.array(grp)
    n, nG = len(grp), int(grp.max()) + 1
    key = np.sort(grp.astype(np.uint64) << np.uint64(32) | np.arange(n, dtype=np.uint64))
    start = np.array([seg.start(key.ctypes.data, n, g) for g in range(nG + 1)], np.int32)
    gs, ge = start[:-1].copy(), start[1:].copy()
    assert np.all(np.diff(start) >= 0) and start[0] == 0 and start[-1] == n
    assert np.array_equal(ge - gs, np.bincount(grp, minlength=nG))
    for t in range(n):
        assert seg.at(gs.ctypes.data, ge.ctypes.data, nG, t) == int(key[t] >> np.uint64(32))


def test_random_ids(seg):
    rng = np.random.default_rng(6)
    for _ in range(50):
        n = int(rng.integers(1, 300))
        grp = rng.choice(rng.choice(60, int(rng.integers(1, 20))), n)
        test_members_and_starts(seg, grp)
