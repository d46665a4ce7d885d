"""The incremental sort where its 32-bit step number wraps: the builds around the
wrap are the radix sort's, in one launch and in two, with most cells never entered
before."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [2 ** 32 - 4, 2 ** 32 - 1])
@pytest.mark.parametrize("cells,n", [(9, 2000), (64, 5000)])
def test_builds_around_the_wrap(cells, n, first, monkeypatch):
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=3)
    rng = np.random.default_rng(n)
    d.cell_size, d.dt, d.wall_mask = 0.1, 1e-3, 0
    for a in range(3):
        d.gravity[a] = 0.0
        d.grid_lo[a], d.grid_hi[a] = -0.1, 0.1 * cells + 0.1
    arrs = {k: rng.uniform(0.1, 0.1 * cells - 0.1, n) for k in "xyz"}
    arrs.update({k: rng.uniform(-3.0, 3.0, n) for k in ("vx", "vy", "vz")})
    arrs["radius"] = np.full(n, 0.03)   # a step of at most 0.0052 stays within a quarter of it
    arrs["mass"] = np.full(n, 1e3)      # and contacts push too little to matter
    got = {}
    for policy, epoch in (("incremental", first), ("radix", 0)):
        monkeypatch.setenv("PRESTIGE_SORT", policy)
        monkeypatch.setenv("PRESTIGE_EPOCH", str(epoch))
        builds = []
        with pa.Context(d) as ctx:
            upload_all(ctx, arrs)
            for _ in range(7):
                ctx.step(1)   # counts and lists the moved spheres under its epoch
                ctx.neighbors_build()
                builds.append(ctx.neighbors_download())
                ctx.step(1)   # from a build of its own
                builds.append({k: ctx.download(k) for k in ("x", "vz")})
        got[policy] = builds
    moved = 0
    for a, b in zip(got["incremental"], got["radix"]):
        assert a.keys() == b.keys()
        for k in a:
            assert np.array_equal(a[k], b[k]), k
        moved += int("perm" in a and np.any(a["perm"] != np.arange(n)))
    assert moved
