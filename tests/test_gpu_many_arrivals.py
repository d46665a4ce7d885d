"""More particles entering one cell in one step than a list takes of runaways, all of
them within the time step's bound: no error, and the radix sort's build."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [pa.F64, pa.MIXED])
@pytest.mark.parametrize("cells", [3, 70])   # a build of one launch, and of two
def test_coincident_spheres_cross_together(cells, precision, monkeypatch):
    """70,000 spheres at one point (which do not touch: contacts need a distance) move over a cell's face, a few
    at a time the other way."""
    n, back = 70000, 300
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=3, precision=precision)
    d.cell_size, d.dt, d.wall_mask = 1.0, 1e-3, 0
    for a in range(3):
        d.gravity[a], d.grid_lo[a], d.grid_hi[a] = 0.0, 0.0, float(cells)
    arrs = {k: np.full(n, 0.5) for k in "xyz"}
    arrs.update(vx=np.full(n, 4.0), vy=np.zeros(n), vz=np.zeros(n), radius=np.full(n, 0.1), mass=np.full(n, 1.0))
    arrs["x"][:] = 0.998
    arrs["x"][::n // back], arrs["vx"][::n // back], arrs["y"][::n // back] = 1.002, -4.0, 0.9   # out of their reach
    got = {}
    for policy in ("incremental", "radix"):
        monkeypatch.setenv("PRESTIGE_SORT", policy)
        with pa.Context(d) as ctx:
            upload_all(ctx, arrs)
            out = []
            for _ in range(2):
                ctx.step(1)
                ctx.neighbors_build()
                out.append(ctx.neighbors_download())
                out[-1].update({k: ctx.download(k) for k in ("x", "vx")})
        got[policy] = out
    for a, b in zip(got["incremental"], got["radix"]):
        for k in a:
            assert np.array_equal(a[k], b[k]), k
    moved = int(np.count_nonzero(arrs["vx"] > 0.0))
    assert moved > 65536
    assert list(got["incremental"][0]["lb"][:3]) == [0, n - moved, n]
