"""The term of a list entry (skg_hit.h, compiled for the host): an entry that the exact test drops adds
nothing to a mover's sums, wherever it lies, and where the step multiplies by zero instead every
separation is finite."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skid_amd", "csrc")


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("hit")
    src, so = d / "hit.cpp", d / "libhit.so"
    src.write_text('#define SKG_HIT_FN static inline\n#include "skg_hit.h"\n'
                   'extern "C" float term(int hit, float d, float f) { return hit_term(hit != 0, d, f); }\n'
                   'extern "C" int far(float x, float y, float z) { return far_off(x, y, z); }\n')
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, "-o", str(so), str(src)],
                   check=True)
    h = ctypes.CDLL(str(so))
    h.term.argtypes, h.term.restype = [ctypes.c_int, ctypes.c_float, ctypes.c_float], ctypes.c_float
    h.far.argtypes, h.far.restype = [ctypes.c_float] * 3, ctypes.c_int
    return h


@pytest.fixture(scope="module")
def hit_term(lib):
    return lib.term


FAR = [np.nan, np.inf, -np.inf, 3.0e38, -3.0e38]


@pytest.mark.parametrize("d", FAR + [0.0, -0.25])
@pytest.mark.parametrize("f", FAR + [0.0, -2.5])
def test_dropped_entry_adds_zero(hit_term, d, f):
    t = np.float32(hit_term(0, d, f))
    assert t == 0 and not np.signbit(t)


def test_step_with_a_far_entry_equals_the_walk(hit_term):
    """One mover's marks in order: balls that hold it, balls that do not, and entries whose mark comes from an
    unordered test alone.  The sum is that of the hits, bit for bit."""
    rng = np.random.default_rng(3)
    n = 64
    pos = rng.uniform(-0.2, 0.2, n).astype(np.float32)
    ball2 = rng.uniform(0.0, 0.05, n).astype(np.float32)
    f = rng.standard_normal(n).astype(np.float32)
    pos[[5, 17, 40, 63]], ball2[[5, 17, 40, 63]] = [np.nan, np.inf, -np.inf, 3.0e38], np.inf
    f[[5, 17, 40, 63]] = 0.0
    with np.errstate(over="ignore", invalid="ignore"):
        d = pos - np.float32(0.01)
        hit = (d * d < ball2) & np.isfinite(d * d)
    assert 8 < hit.sum() < 56 and not hit[[5, 17, 40, 63]].any()
    steps, walk = 0.0, 0.0
    for i in range(n):
        steps += hit_term(int(hit[i]), float(d[i]), float(f[i]))
        if hit[i]:
            walk += float(d[i] * f[i])
    assert steps == walk


def test_near_positions_have_finite_separations(lib):
    """No position that passes as near lies so far from another one that their separation overflows, nor its
    sum with a period's shift (a replica and its source are near, so the shift is at most twice as far)."""
    edge = [0.0, 0.5, -0.5, 1e20, -1e20, 0.99e37, -0.99e37, 1.01e37, -3.4e38, np.inf, -np.inf, np.nan]
    near = [np.float32(v) for v in edge if not lib.far(v, 0.0, 0.0)]
    assert len(near) == 7
    for a in near:
        for b in near:
            assert np.isfinite(a - b)
            assert np.isfinite((a - b) + np.float32(2) * near[-2]) and np.isfinite((a - b) + np.float32(2) * near[-1])
    for v in edge[7:]:
        assert lib.far(v, 0, 0) and lib.far(0, v, 0) and lib.far(0, 0, v)
