"""Contexts without the incremental sort's lists and counts per cell, as where these
do not fit: the same builds and states, and no more memory for a grid of billions of
cells than its cell table takes."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all
from test_zz_no_alloc import hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene,precision", [(pa.SCENE_DEM_POUR, pa.F64), (pa.SCENE_DEM_POUR, pa.MIXED), (pa.SCENE_DAM_BREAK, pa.F64),
                                             (pa.SCENE_DAM_BREAK, pa.F32), (pa.SCENE_DAM_BREAK, pa.MIXED)])
def test_same_steps(scene, precision, monkeypatch):
    d, arrs = make_scene(scene, n_target=3000, dx=0.01, seed=5, precision=precision)
    got = {}
    for policy in ("keys", "incremental"):
        monkeypatch.setenv("PRESTIGE_SORT", policy)
        out = []
        with pa.Context(d) as ctx:
            upload_all(ctx, arrs if scene == pa.SCENE_DEM_POUR else {k: arrs[k] for k in ("x", "y", "z", "vx", "vy", "vz")})
            for steps in (1, 20, 3):
                ctx.step(steps)
                ctx.neighbors_build()
                out.append(ctx.neighbors_download())
                out[-1].update({k: ctx.download(k) for k in ("x", "vz")})
        got[policy] = out
    for a, b in zip(got["keys"], got["incremental"]):
        for k in a:
            assert np.array_equal(a[k], b[k]), k


def _free():
    left, total = C.c_size_t(), C.c_size_t()
    assert hip().hipMemGetInfo(C.byref(left), C.byref(total)) == 0
    return left.value


def test_grid_of_billions_of_cells():
    """3.9e9 cells: the table is 15.6 GB; lists and counts would be 78 more, over a quarter of the device."""
    n = 500
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=3)
    d.cell_size, d.dt, d.wall_mask, d.kn, d.kt = 0.1, 1e-3, 0, 1e-2, 1e-3
    rng = np.random.default_rng(0)
    arrs = {k: rng.uniform(0.1, 1.4, n) for k in "xyz"}
    arrs.update({k: rng.uniform(-4.0, 4.0, n) for k in ("vx", "vy", "vz")})
    arrs["radius"], arrs["mass"] = np.full(n, 0.03), np.full(n, 1e3)
    got = []
    for dims in ((15, 15, 15), (1560, 1580, 1582)):
        for a in range(3):
            d.gravity[a], d.grid_lo[a], d.grid_hi[a] = 0.0, 0.0, 0.1 * dims[a]
        before = _free()
        with pa.Context(d) as ctx:
            took = before - _free()
            upload_all(ctx, arrs)
            ctx.step(3)
            got.append({k: ctx.download(k) for k in ("x", "y", "z", "vx", "wx")})
    assert took < 20e9
    for k in got[0]:
        assert np.array_equal(got[0][k], got[1][k]), k
