"""Removal with every member resident (k_unb_res), at the group sizes where its classes and slots
end, with and without kdSubPot, against the FP64 restatement of kdUnbind."""
import numpy as np
import pytest

from oracle import oracle as O
from skid_amd import gen, skg

pytestmark = pytest.mark.gpu

SIZES = [64, 65, 128, 511, 512, 513, 1025, 2047, 2048, 2049, 4097, 8192, 8193]


def hot_groups(seed):
    rng = np.random.default_rng(seed)
    n = sum(SIZES)
    pos, vel, grp = np.empty((n, 3)), np.empty((n, 3)), np.empty(n, np.int32)
    mass = rng.uniform(0.5, 1.5, n) / n
    a = 0
    for g, m in enumerate(SIZES):
        r200 = float(gen.r200_of(m / n))
        c = rng.uniform(-0.5, 0.5, 3)                # some spheres lie across a face
        pos[a:a + m] = c + gen._iso_dirs(rng, m) * (gen.nfw_radii(rng, m, 8.0) * r200)[:, None]
        vel[a:a + m] = rng.normal(0.0, np.sqrt(1.6 * m / n / (2 * r200)), (m, 3))
        grp[a:a + m] = g + 1
        a += m
    o = rng.permutation(n)
    return gen._wrap(pos[o]), vel[o].astype(np.float32), mass[o].astype(np.float32), grp[o]


@pytest.mark.parametrize("gas", [False, True])
def test_removal_matches_fp64_at_the_class_edges(gas):
    pos, vel, mass, grp = hot_groups(17)
    n = len(grp)
    soft = np.full(n, 0.0288 * n ** (-1.0 / 3.0), np.float32)
    box = gen.Box(pos=pos, vel=vel, mass=mass, soft=soft, temp=np.zeros(n, np.float32),
                  n_gas=n if gas else 0, n_dark=0 if gas else n)
    fs, fc = gen.config5_cosmology()
    ctx = skg.Context(box, skg.make_params(0.01, 32, period=1.0, z=0.5, fShift=fs, fCosmo=fc))
    ng = ctx.set_groups(grp)
    nu = ctx.unbind()
    got, _ = ctx.groups()
    cat = ctx.catalogue(ng)
    ctx.close()
    want = O.unbind_f64(pos, vel, mass, soft, grp, None, fshift=fs, fcosmo=fc, z=0.5, sub_pot=not gas)
    assert nu == int((got == 0).sum()) and nu > 0
    for g, m in enumerate(SIZES, 1):
        mem = grp == g
        assert np.mean((got[mem] > 0) == (want[mem] > 0)) >= 0.999, (g, m)
        left = got == g
        assert cat["nmembers"][g] == left.sum(), (g, m)
        if left.sum() == 0:
            continue
        w = mass[left].astype(np.float64)
        # FP64 sums of fp32 products, rounded once to fp32, from which the removed members were taken off
        assert abs(cat["mass"][g] - w.sum()) <= 4e-7 * mass[mem].sum(), (g, m)
        v = (w[:, None] * vel[left]).sum(0) / w.sum()
        scale = np.abs(vel[mem]).max() * mass[mem].sum() / w.sum()
        assert np.all(np.abs(cat["vcm"][g] - v) <= 4e-7 * scale), (g, m)
