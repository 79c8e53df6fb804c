"""The register kNN (compensated mode, up to 128 neighbours): radii, neighbour sets and their order of
ties equal a brute-force search in the same fp32 arithmetic, bit for bit."""
import numpy as np
import pytest

from skid_amd import gen, skg

pytestmark = pytest.mark.gpu


def points(kind, n, seed):
    rng = np.random.default_rng(seed)
    if kind == "lattice":                               # shells of exact ties, more than eight at once
        m = int(np.ceil(n ** (1 / 3)))
        g = (np.arange(m) + 0.5) / m - 0.5
        x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)[:n]
    elif kind == "coincident":                          # more points on one spot than neighbours
        x = rng.uniform(-0.5, 0.5, (n, 3))
        x[: n // 2] = x[0]
    else:
        c = rng.uniform(-0.5, 0.5, (max(1, n // 200), 3))
        x = c[rng.integers(0, len(c), n)] + 0.02 * rng.standard_normal((n, 3)) * rng.random((n, 1))
        x[::5] = rng.uniform(-0.5, 0.5, (len(x[::5]), 3))
        x -= np.floor(x + 0.5)
    pos = x.astype(np.float32)
    pos[pos <= -0.5] = 0.5
    z = np.zeros(n, np.float32)
    return gen.Box(pos=pos, vel=np.zeros((n, 3), np.float32), mass=np.full(n, 1 / n, np.float32), soft=z + 0.01,
                   temp=z, n_gas=0, n_dark=n)


def brute(pos, k, periodic):
    d2 = np.zeros((len(pos), len(pos)), np.float32)
    one, half = np.float32(1), np.float32(0.5)
    for a in range(3):
        q, p = pos[:, None, a], pos[None, :, a]
        d = q - p
        if periodic:                                    # the image is taken on the query's side
            d = np.where(d > half, (q - one) - p, np.where(d < -half, (q + one) - p, d))
        d2 = d2 + d * d if a else d * d
    idx = np.argsort(d2, axis=1, kind="stable")[:, :k]  # ties: smallest index first
    return idx, np.take_along_axis(d2, idx, 1)


@pytest.mark.parametrize("kind,n,k,B,periodic", [
    ("clumps", 2, 2, 16, False),
    ("clumps", 64, 64, 16, True),         # every point a neighbour
    ("clumps", 65, 31, 64, True),
    ("clumps", 1000, 32, 16, True),
    ("clumps", 1001, 33, 24, False),      # leaves not a power of two
    ("clumps", 2049, 64, 7, True),
    ("clumps", 2049, 65, 100, True),      # two windows per leaf
    ("clumps", 3000, 128, 1, True),       # more leaves than are kept for the second visit
    ("clumps", 3000, 128, 1, False),
    ("lattice", 1728, 32, 16, True),
    ("lattice", 1728, 64, 16, True),
    ("lattice", 2000, 100, 16, False),
    ("coincident", 600, 32, 16, True),
    ("coincident", 600, 128, 16, False),
])
def test_neighbours_equal_brute_force(kind, n, k, B, periodic):
    box = points(kind, n, 3 * n + k)
    P = skg.make_params(0.01, k, nBucket=B, period=1.0 if periodic else None)
    ctx = skg.Context(box, P)
    b2, rho, _ = ctx.density()
    nb, d2 = ctx.neighbors()
    idx, ref = brute(box.pos, k, periodic)
    assert np.array_equal(b2, ref[:, -1])
    assert np.array_equal(d2, ref)
    assert np.array_equal(nb, idx)


def test_batched_boxes_keep_to_themselves():
    """Small boxes that share leaves and windows: each one's neighbours are its own."""
    sizes = [40, 33, 200, 65, 1000, 34]
    boxes = [points("lattice" if b == 4 else "clumps", n, b) for b, n in enumerate(sizes)]
    ctx = skg.BatchContext(boxes, skg.make_params(0.01, 33, period=1.0), np.full(len(sizes), 0.01, np.float32))
    ctx.density()
    nb, d2 = ctx.neighbors()
    for b, box in enumerate(boxes):
        lo, hi = ctx.offsets[b], ctx.offsets[b + 1]
        idx, ref = brute(box.pos, 33, True)
        assert np.array_equal(d2[lo:hi], ref), b
        assert np.array_equal(nb[lo:hi] - lo, idx), b
