"""The incremental sort against the full radix sort: the same permutation, keys,
cell table and state after steps in which slots move up, down and within a
tile of cells, in grids of one cell to several tiles, and its bound on the
slots one cell takes in a step."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all

pytestmark = pytest.mark.gpu


def _builds(d, arrs, policy, steps, monkeypatch):
    monkeypatch.setenv("PRESTIGE_SORT", policy)
    out = []
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        for _ in range(steps):
            try:
                ctx.step(1)
            except pa.PrestigeError as e:
                assert e.name == "E_CFL", str(e)   # these spheres outrun the contact step on purpose
            ctx.neighbors_build()
            out.append(ctx.neighbors_download())
        state = {k: ctx.download(k) for k in ("x", "y", "z", "vx", "wz")}
    return out, state


@pytest.mark.parametrize("precision", [pa.F64, pa.MIXED])
@pytest.mark.parametrize("cells,n,move", [(1, 100, 0.3), (2, 257, 0.4), (5, 3000, 0.2), (23, 20000, 0.02), (23, 20000, 0.5)])
def test_same_build_as_the_radix_sort(cells, n, move, precision, monkeypatch):
    """n spheres in cells^3 cells, each moving up to `move` cells a step; every fifth starts fixed in the state
    (id >= n_moving)."""
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=3, precision=precision)
    rng = np.random.default_rng(cells * n)
    d.n_moving = n - n // 5
    d.cell_size = 0.1
    d.dt = 1e-3
    for a in range(3):
        d.gravity[a] = 0.0
        d.grid_lo[a], d.grid_hi[a] = -0.1, 0.1 * cells + 0.1   # a margin of cells that start empty
    d.wall_mask = 0
    arrs = {k: rng.uniform(0.0, 0.1 * cells, n) for k in "xyz"}
    arrs.update({k: rng.uniform(-move, move, n) * 0.1 / 4 / d.dt for k in ("vx", "vy", "vz")})
    arrs["radius"] = np.full(n, 1e-6)
    arrs["mass"] = np.full(n, 1e-6)
    inc, s1 = _builds(d, arrs, "incremental", 4, monkeypatch)
    rad, s2 = _builds(d, arrs, "radix", 4, monkeypatch)
    for step, (a, b) in enumerate(zip(inc, rad)):
        for k in ("keys", "perm", "ids", "lb"):
            assert np.array_equal(a[k], b[k]), (step, k)
    for k in s1:
        assert np.array_equal(s1[k], s2[k]), k
    assert cells == 1 or any(np.any(g["perm"] != np.arange(n)) for g in inc)


@pytest.mark.parametrize("cells", [61, 62])
def test_largest_grid_of_one_launch_and_the_next(cells, monkeypatch):
    """63^3 cells are 245 tiles, each block scans them with a thread each; 64^3 and the table's last entry are 257."""
    test_same_build_as_the_radix_sort(cells, 30000, 0.3, pa.F64, monkeypatch)


def test_counts_that_no_build_took(monkeypatch):
    """An upload after a step drops what the step counted: the builds after it start from cleared counts."""
    d, arrs = make_scene(pa.SCENE_DEM_POUR, n_target=3000, seed=5)
    out = {}
    for policy in ("incremental", "radix"):
        monkeypatch.setenv("PRESTIGE_SORT", policy)
        got = []
        with pa.Context(d) as ctx:
            upload_all(ctx, {**arrs, "vx": np.full(len(arrs["x"]), 0.2)})
            for steps in (1, 2, 3):
                ctx.step(steps)
                ctx.upload("x", ctx.download("x"))
                ctx.step(2)
                ctx.neighbors_build()
                got.append(ctx.neighbors_download())
        out[policy] = got
    for a, b in zip(out["incremental"], out["radix"]):
        for k in ("keys", "perm", "ids", "lb"):
            assert np.array_equal(a[k], b[k]), k


def test_a_runaway_into_one_cell_stays_bounded():
    """70,000 spheres jump into one cell in one step: the error names the runaway, no sphere is lost, and at
    most 65,536 of them changed cell."""
    n = 70000
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=3)
    d.cell_size, d.dt, d.wall_mask = 1.0, 1e-3, 0
    d.grid_lo[0], d.grid_hi[0] = 0.0, 2.0
    for a in (1, 2):
        d.grid_lo[a], d.grid_hi[a] = 0.0, 1.0
    for a in range(3):
        d.gravity[a] = 0.0
    rng = np.random.default_rng(0)
    arrs = {k: rng.uniform(0.1, 0.9, n) for k in "xyz"}
    arrs.update(vx=np.full(n, 1.0 / d.dt), vy=np.zeros(n), vz=np.zeros(n), radius=np.full(n, 1e-7), mass=np.full(n, 1.0))
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        with pytest.raises(pa.PrestigeError) as e:
            ctx.step(1)
        assert e.value.name == "E_CFL"
        assert np.array_equal(ctx.download("x"), arrs["x"] + d.dt * arrs["vx"])
        ctx.neighbors_build()
        g = ctx.neighbors_download()
    assert np.array_equal(np.sort(g["ids"]), np.arange(n))
    assert list(g["lb"]) == [0, n - 65536, n]
