"""Wall springs: kept while a sphere touches a wall, forgotten when it leaves,
and without a trace of an earlier contact when it comes back or the positions
are set again."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, oracle_state, upload_all

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "wx", "wy", "wz")


def _between_plates(n):
    """Spheres that do not meet, bouncing between two plates little more than a diameter apart and off side
    walls; every seventh is fixed."""
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=4, seed=0)
    side = int(np.ceil(np.sqrt(n)))
    r, gap = 0.01, 0.05
    d.n_particles = n
    d.n_moving = n - n // 7
    d.cell_size = 0.05
    d.wall_mask = 63
    size = (side * gap, side * gap, 2.02 * r)
    for a in range(3):
        d.gravity[a] = 0.0
        d.grid_lo[a], d.grid_hi[a], d.wall_lo[a], d.wall_hi[a] = -0.05, size[a] + 0.05, 0.0, size[a]
    rng = np.random.default_rng(n)
    k = np.arange(n)
    pos = np.stack([(k % side + 0.5) * gap, (k // side + 0.5) * gap, np.full(n, 1.01 * r)], 1)
    pos[k % side == 0, 0] = 1.005 * r
    vel = np.concatenate([rng.uniform(-0.3, 0.3, (n, 2)), rng.choice([-1.0, 1.0], (n, 1)) * rng.uniform(0.5, 1.0, (n, 1))], 1)
    arrs = {c: np.ascontiguousarray(pos[:, i]) for i, c in enumerate("xyz")}
    arrs.update({c: np.ascontiguousarray(vel[:, i]) for i, c in enumerate(("vx", "vy", "vz"))})
    arrs["radius"] = np.full(n, r)
    arrs["mass"] = np.full(n, 0.01)
    return d, arrs


@pytest.mark.parametrize("n", [1, 15, 64, 500])
def test_touch_leave_and_touch_again(n):
    d, arrs = _between_plates(n)
    st = oracle_state(d, arrs)
    touching = []
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        for _ in range(30):
            assert st.step(10) == 0
            ctx.step(10)
            z = st.get("z")[: d.n_moving]
            touching.append(np.where(z < 0.01, -1, np.where(z > 0.0102, 1, 0)))
        for k in FIELDS:
            assert np.array_equal(ctx.download(k), st.get(k)), k
        # set again, spins too: as if new
        upload_all(ctx, arrs)
        for k in ("wx", "wy", "wz"):
            ctx.upload(k, np.zeros(n))
        ctx.step(25)
        again = {k: ctx.download(k) for k in FIELDS}
    t = np.array(touching)
    assert (t == 1).any() and (t == -1).any() and (t == 0).any()
    fresh = oracle_state(d, arrs)
    assert fresh.step(25) == 0
    for k in FIELDS:
        assert np.array_equal(again[k], fresh.get(k)), k
