"""The wavefront-per-point cover kernel (scatter density and Denmax step of small point sets)
against FP64 brute force, at the leaf sizes and point counts where its rounds have edges."""
import itertools

import numpy as np
import pytest

from skid_amd import gen, skg

pytestmark = pytest.mark.gpu


def clumps(n, seed):
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.5, 0.5, (max(1, n // 300), 3))
    x = c[rng.integers(0, len(c), n)] + 0.03 * rng.standard_normal((n, 3)) * rng.random((n, 1))
    x[::4] = rng.uniform(-0.5, 0.5, (len(x[::4]), 3))
    pos = (x - np.floor(x + 0.5)).astype(np.float32)
    pos[pos <= -0.5] = 0.5
    m = (rng.uniform(0.5, 1.5, n) / n).astype(np.float32)
    z = np.zeros(n, np.float32)
    return gen.Box(pos=pos, vel=np.zeros((n, 3), np.float32), mass=m, soft=z + 0.01, temp=z, n_gas=0, n_dark=n)


def brute(pos, mass, b2, periodic):
    """FP64 density, and per point the gradient of the scatter field and the sum of its terms' sizes.
    A ball of more than half a period can hold a point through several of its images."""
    x, m, h = pos.astype(np.float64), mass.astype(np.float64), 0.5 * np.sqrt(b2.astype(np.float64))
    d0 = x[None, :, :] - x[:, None, :]                 # [point, scatterer]
    near = -np.round(d0) if periodic else np.zeros_like(d0)
    shifts = [np.zeros(3)]
    if periodic and h.max() > 0.25:
        shifts = [np.array(s, float) for s in itertools.product((-1, 0, 1), repeat=3)]
    rho, a, size = np.zeros(len(x)), np.zeros_like(x), np.zeros_like(x)
    for s in shifts:
        image = near + s
        d = d0 + image
        # a ball holds a point by the fp32 distance to the (rounded) image, strictly
        d32 = (pos[None, :, :] + image.astype(np.float32)) - pos[:, None, :]
        holds = d32[..., 0] * d32[..., 0] + d32[..., 1] * d32[..., 1] + d32[..., 2] * d32[..., 2] < b2[None, :]
        q = np.sqrt((d * d).sum(2)) / h[None, :]
        w = np.where(q < 1, 1 + q * q * (0.75 * q - 1.5), 0.25 * np.clip(2 - q, 0, None) ** 3)
        W = 0.5 * w / (np.pi * h[None, :] ** 3)
        rho += np.where(holds, W * m[None, :], 0.0).sum(1)
        if not s.any():
            rho += (W * m[:, None]).sum(0)             # the gather half: nearest images
        g = np.where(q < 1, 2.25 * q - 3, -0.75 * np.clip(2 - q, 0, None) ** 2 / np.maximum(q, 1e-30))
        t = d * np.where(holds, m / (np.pi * h ** 5) * g, 0.0)[:, :, None]
        a += t.sum(1)
        size += np.abs(t).sum(1)
    return rho, a, size


@pytest.mark.parametrize("n,k,B,plain,periodic", [
    (64, 8, 16, False, True),         # one full wavefront's worth of points
    (33, 4, 64, False, True),         # one leaf
    (65, 8, 1, True, False),          # one entity per leaf, one more point than a wavefront
    (1000, 32, 3, False, True),       # leaf size not a power of two
    (1000, 33, 24, True, False),
    (2049, 32, 16, True, False),
    (2049, 32, 32, False, True),
    (4099, 64, 64, False, True),
    (4099, 32, 128, False, True),     # leaves of several rounds
    (4099, 256, 1, False, True),      # more opened nodes than the frontier holds
])
def test_wave_per_point_against_fp64(n, k, B, plain, periodic):
    box = clumps(n, 7 * n + B)
    tau = 0.16 * n ** (-1.0 / 3.0)
    P = skg.make_params(tau, k, nBucket=B, period=1.0 if periodic else None,
                        accumulate=skg.SKG_ACC_PLAIN if plain else skg.SKG_ACC_COMPENSATED)
    ctx = skg.Context(box, P)
    b2, rho, _ = ctx.density()
    r64, a, size = brute(box.pos, box.mass, b2, periodic)
    assert np.max(np.abs(rho - r64) / r64) < 1e-5
    ctx.init_move()
    ctx.move_first()
    got = ctx.moved().astype(np.float64)
    ctx.close()
    # the step is fStep along -a: its error is a's direction error (8e-6 of the terms' sizes, the fp32
    # terms' rounding) times fStep, and the position's own rounding
    step = float(P.fStep)
    na = np.sqrt((a * a).sum(1))
    want = box.pos.astype(np.float64) - step * a / np.maximum(na, 1e-300)[:, None]
    d = got - want
    if periodic:
        d -= np.round(d)
    err = np.sqrt((d * d).sum(1))
    tol = 2e-7 + step * np.minimum(2.1, 8e-6 * np.sqrt((size * size).sum(1)) / np.maximum(na, 1e-300))
    alone = size.sum(1) == 0                         # in no ball but its own: stays
    tol[alone] = np.inf
    assert np.all(err <= tol), (int((err > tol).sum()), float(np.max(err / tol)))
    assert np.array_equal(got[alone], box.pos[alone].astype(np.float64))
