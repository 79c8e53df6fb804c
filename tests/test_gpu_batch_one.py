"""A batch of one box with its own tau is that box run alone with that tau."""
import numpy as np
import pytest

from skid_amd import gen, skg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("factor", [0.5, 3.0])
def test_one_box_takes_its_own_tau(factor):
    n = 8000
    box, tau = gen.config4_box(n, 4), float(np.float32(gen.config4_tau(n)))
    kw = dict(nSmooth=32, period=1.0, fDensMin=40.0)     # a density floor leaves particles to the scoop
    batch = skg.BatchContext([box], skg.make_params(factor * tau, **kw), np.array([tau], np.float32))
    alone = skg.Context(box, skg.make_params(tau, **kw))
    got = []
    for ctx in (batch, alone):
        ctx.density()
        ctx.move_loop(max_blocks=2000)
        fof, nfof = ctx.fof()
        ctx.microsteps()
        ctx.centers()
        nunb = ctx.unbind()
        ctx.too_small()
        g, ng = ctx.groups()
        got.append((fof.copy(), nfof, nunb, g.copy(), ng))
        ctx.close()
    assert got[1][4] > 2 and got[1][2] > 0
    for a, b in zip(*got):
        assert np.array_equal(a, b)
