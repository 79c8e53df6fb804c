"""Entity lists of a move block in batched contexts: tiles of 64 movers that hold two boxes, with
movers that leave their tile by crossing a face, against the walk without lists, bit for bit."""
import numpy as np
import pytest

from skid_amd import gen, skg

pytestmark = pytest.mark.gpu

# movers of the next box in a box's last tile: 1, 63, 2, none, 31, 1, 3
LANES = [1, 63, 2, 0, 31, 1, 3]
TAU = 0.02


def corner_boxes():
    """Boxes of about a thousand particles; in each a clump around the point where all faces meet, so that the
    first movers along the curve step across faces from the first block on.  Every second box is a hundred times
    as heavy, so its densities and thresholds lie above its neighbours'."""
    rng = np.random.default_rng(11)
    boxes, total = [], 0
    for b in range(len(LANES) + 1):
        n = 640 + 64 * b
        if b < len(LANES):
            n += (-LANES[b] - total - n) % 64        # the box ends LANES[b] lanes short of a whole tile
            total += n
        x = rng.uniform(-0.5, 0.5, (n, 3))
        x[: n // 4] = 0.5 + 0.012 * rng.standard_normal((n // 4, 3))
        x[:8] = -0.5 + 0.0004 * (1 + np.arange(8))[:, None]
        x = x[rng.permutation(n)]
        pos = (x - np.floor(x + 0.5)).astype(np.float32)
        pos[pos <= -0.5] = 0.5
        z = np.zeros(n, np.float32)
        m = np.full(n, (100.0 if b % 2 else 1.0) / n, np.float32)
        boxes.append(gen.Box(pos=pos, vel=np.zeros((n, 3), np.float32), mass=m, soft=z + 0.01, temp=z, n_gas=0,
                             n_dark=n))
    return boxes


def blocks(monkeypatch, env, acc, steps=4):
    """Positions, live entities and active movers of every box after each of the first blocks."""
    for k in ("SKG_TILE_LISTS", "SKG_TILE_CAP", "SKG_GRAPH"):
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setenv("SKG_COVER_SUB_MAX", "0")         # every step takes the lane-per-mover kernel
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    boxes = corner_boxes()
    ctx = skg.BatchContext(boxes, skg.make_params(TAU, 32, period=1.0, accumulate=acc),
                           np.full(len(boxes), TAU, np.float32))
    ctx.density()
    ctx.init_move()
    ctx.move_first()
    out = []
    for _ in range(steps):
        ctx.move_block()
        a, s = ctx.box_counts()
        out.append((ctx.moved(), np.array(s), np.array(a)))
    ctx.close()
    return out


@pytest.mark.parametrize("acc", [skg.SKG_ACC_COMPENSATED, skg.SKG_ACC_PLAIN])
@pytest.mark.parametrize("env", [{}, {"SKG_TILE_CAP": "64"}, {"SKG_GRAPH": "1", "SKG_TILE_CAP": "64"},
                                 {"SKG_TILE_LISTS": "2"}])
def test_tiles_of_two_boxes_equal_the_walk(env, acc, monkeypatch):
    want = blocks(monkeypatch, {"SKG_TILE_LISTS": "0"}, acc)
    got = blocks(monkeypatch, env, acc)
    assert want[0][2].sum() > 0
    for i, (w, g) in enumerate(zip(want, got)):
        assert np.array_equal(w[1], g[1]), i              # live entities: each box's own thresholds
        assert np.array_equal(w[2], g[2]), i
        differ = np.flatnonzero((w[0] != g[0]).any(1))
        assert differ.size == 0, (i, differ.size)
