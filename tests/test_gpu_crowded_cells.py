"""First builds with one crowded cell: the radix sort's result at any occupancy, also
around the line where a build leaves the counting sort, and particles that all lie
outside the grid, whose error must not cost more than a build."""
from __future__ import annotations

import time

import numpy as np
import pytest

import prestige_amd as pa

pytestmark = pytest.mark.gpu


def _context(n, dims, precision=pa.F64):
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.precision = precision
    d.cell_size = 1.0
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, float(dims[a])
    return pa.Context(d)


def _build(policy, pts, dims, precision, monkeypatch):
    monkeypatch.setenv("PRESTIGE_SORT", policy)
    out = []
    with _context(len(pts), dims, precision) as ctx:
        for order in (pts, np.ascontiguousarray(pts[::-1])):   # the second from the order the first left
            for a, k in enumerate("xyz"):
                ctx.upload(k, np.ascontiguousarray(order[:, a]))
            ctx.neighbors_build()
            out.append(ctx.neighbors_download())
            out[-1].update({k: ctx.download(k) for k in "xyz"})
    return out


@pytest.mark.parametrize("precision", [pa.F64, pa.F32])
@pytest.mark.parametrize("n,crowd", [(2048, 2048), (2049, 2049), (2100, 2048), (5000, 2048), (5000, 2049), (30000, 20000), (200000, 120000)])
def test_same_build_as_the_radix_sort(n, crowd, precision, monkeypatch):
    rng = np.random.default_rng(n + crowd)
    dims = (20, 18, 16)
    pts = rng.uniform(0.0, 1.0, (n, 3)) * dims * 0.999
    pts[:, 0] = np.where(pts[:, 0] < 1.0, pts[:, 0] + 1.0, pts[:, 0])   # none but the crowd in cell x = 0
    pts[rng.permutation(n)[:crowd]] = rng.uniform(0.0, 0.9, (crowd, 3)) + [0.0, 7.0, 9.0]
    pts = pts.astype(np.float32).astype(np.float64)
    got, want = _build("counting", pts, dims, precision, monkeypatch), _build("radix", pts, dims, precision, monkeypatch)
    assert int(np.max(np.diff(want[0]["lb"].astype(np.int64)))) == crowd
    for g, w in zip(got, want):
        for k in g:
            assert np.array_equal(g[k], w[k]), k


def test_all_particles_outside_the_grid():
    """400,000 particles in wrong units: the error, in the time of a few builds (17 ms by the lists of one cell,
    below 1 by the radix sort), and the context builds again once they are right."""
    n, dims = 400000, (100, 100, 100)
    pts = np.random.default_rng(0).uniform(0.0, 99.9, (n, 3))
    with _context(n, dims) as ctx:
        took = []
        for _ in range(3):
            ctx.upload("x", pts[:, 0] * 1000.0 + 200.0)
            t = time.perf_counter()
            with pytest.raises(pa.PrestigeError) as e:
                ctx.neighbors_build()
            took.append(time.perf_counter() - t)
            assert e.value.name == "E_DOMAIN"
        assert min(took) < 5e-3
        for a, k in enumerate("xyz"):
            ctx.upload(k, np.ascontiguousarray(pts[:, a]))
        ctx.neighbors_build()
        g = ctx.neighbors_download()
    keys = (np.floor(pts[:, 2]) * 100 + np.floor(pts[:, 1])) * 100 + np.floor(pts[:, 0])
    assert np.array_equal(g["keys"], np.sort(keys))
    # the failed builds left the particles in their order, all with one key
    assert np.array_equal(g["ids"], np.argsort(keys, kind="stable"))
