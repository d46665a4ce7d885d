"""Field transfers: what crosses the pinned block and what the ring of chunks, the checks on
the device, and arrays that outlive later downloads."""

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene

pytestmark = pytest.mark.gpu

BLOCK = (1 << 20) // 8   # values that just fit the pinned block, and a chunk of the ring
RING = 8 * BLOCK


def pairs(n):
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.cell_size = 0.1
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, 1.0
    return pa.Context(d)


@pytest.mark.parametrize("n", [1, 255, BLOCK, BLOCK + 1, 2 * BLOCK - 1, 2 * BLOCK, 2 * BLOCK + 1, RING - 1, RING, RING + 1, 2 * RING + BLOCK + 3])
def test_values_come_back_and_bad_ones_change_nothing(n):
    rng = np.random.default_rng(n)
    x, y, m = rng.random(n), rng.random(n), rng.random(n) + 0.5
    with pairs(n) as c:
        c.upload("x", x)
        c.upload("y", y)
        c.upload("mass", m)
        first = c.download("x")
        view = c.download("y")[n // 2:]
        for bad in (np.nan, np.inf, -np.inf):
            for at in {0, n // 2, n - 1}:
                z = rng.random(n)
                z[at] = bad
                with pytest.raises(pa.PrestigeError, match="non-finite"):
                    c.upload("x", z)
        for _ in range(3):   # blocks are used again, never one that is still in use
            assert np.array_equal(c.download("x"), x)
            assert np.array_equal(c.download("mass"), m)
        c.upload("x", y)
        assert np.array_equal(c.download("x"), y)
    assert np.array_equal(first, x) and np.array_equal(view, y[n // 2:])
    first[:] = 0.0
    assert first.flags.owndata   # ordinary memory of the caller's, which a forked process has too


@pytest.mark.parametrize("n", [300, BLOCK + 1])
def test_sphere_checks(n):
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=4, seed=0)
    d.n_particles = d.n_moving = n
    d.cell_size = 0.1
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a], d.wall_lo[a], d.wall_hi[a] = 0.0, 1.0, 0.0, 1.0
    r, m = np.full(n, 0.05), np.full(n, 2.0)
    with pa.Context(d) as c:
        c.upload("radius", r)     # exactly half a cell is still allowed
        c.upload("mass", m)
        for name, value, text in (("radius", np.nextafter(0.05, 1), "cell_size"), ("radius", 0.0, "radii"),
                                  ("radius", -np.inf, "non-finite"), ("mass", 0.0, "masses"), ("mass", np.nan, "masses")):
            v = (r if name == "radius" else m).copy()
            v[-1] = value
            with pytest.raises(pa.PrestigeError, match=text):
                c.upload(name, v)
        v = r.copy()
        v[0], v[1], v[2] = 1.0, -1.0, np.nan     # the first test in order is the one reported
        with pytest.raises(pa.PrestigeError, match="non-finite"):
            c.upload("radius", v)
        v[2] = 0.05
        with pytest.raises(pa.PrestigeError, match="radii"):
            c.upload("radius", v)
        assert np.array_equal(c.download("radius"), r)
        c.upload("radius", 0.5 * r)
        assert np.array_equal(c.download("radius"), 0.5 * r)
