"""Groups from outside whose ids have gaps: the same groups under consecutive ids give the same result."""
import numpy as np
import pytest

from skid_amd import gen, skg

pytestmark = pytest.mark.gpu


def groups(seed, sizes):
    rng = np.random.default_rng(seed)
    n = sum(sizes) + 500
    pos, vel, grp, a = rng.uniform(-0.5, 0.5, (n, 3)), np.zeros((n, 3)), np.zeros(n, np.int32), 0
    for g, m in enumerate(sizes):
        r200 = float(gen.r200_of(m / n))
        pos[a:a + m] = rng.uniform(-0.5, 0.5, 3) + gen._iso_dirs(rng, m) * (gen.nfw_radii(rng, m, 8.0) * r200)[:, None]
        vel[a:a + m] = rng.normal(0.0, np.sqrt(1.6 * m / n / (2 * r200)), (m, 3))
        grp[a:a + m] = g + 1
        a += m
    o = rng.permutation(n)
    return gen._wrap(pos[o]), vel[o].astype(np.float32), grp[o]


def run(pos, vel, grp, gas):
    n = len(grp)
    box = gen.Box(pos=pos, vel=vel, mass=np.full(n, 1 / n, np.float32),
                  soft=np.full(n, 0.0288 * n ** (-1.0 / 3.0), np.float32), temp=np.zeros(n, np.float32),
                  n_gas=n if gas else 0, n_dark=0 if gas else n)
    fs, fc = gen.config5_cosmology()
    ctx = skg.Context(box, skg.make_params(0.01, 32, period=1.0, z=0.5, fShift=fs, fCosmo=fc))
    ng = ctx.set_groups(grp)
    w, t = ctx.group_energies(ng)
    nu = ctx.unbind()
    ctx.too_small()
    g, ngf = ctx.groups()
    cat = ctx.catalogue(ngf)
    ctx.close()
    return w, t, nu, g, cat


@pytest.mark.parametrize("gas", [False, True])
@pytest.mark.parametrize("ids", [[1, 3, 4, 9], [2, 3, 4, 5], [5, 6, 70, 71]])
def test_missing_ids_change_nothing(ids, gas):
    pos, vel, grp = groups(3, [311, 40, 900, 2500])
    want = run(pos, vel, grp, gas)
    got = run(pos, vel, np.array([0] + ids, np.int32)[grp], gas)
    assert want[2] > 0 and got[2] == want[2]
    for e in (0, 1):
        assert np.array_equal(got[e][ids], want[e][1:])
        assert not np.delete(got[e], ids).any()
    assert np.array_equal(got[3], want[3])                # final ids are consecutive again
    for k in want[4]:
        assert np.array_equal(got[4][k][1:], want[4][k][1:]), k
