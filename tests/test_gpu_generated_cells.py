"""Generated passes over the cell iterator where their scan can go wrong: tile
edges, runs of more candidates than a scan word or the stage holds, and more
tiles than one round over the XCDs.  Whole-number masses, so every sum is exact."""
from __future__ import annotations

import numpy as np
import pytest
from scipy.spatial import cKDTree

import prestige_amd as pa

pytestmark = pytest.mark.gpu


def _run(pos, mass, cell, cutoff, body, precision=pa.F64):
    n = len(pos)
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.precision = precision
    d.cell_size = cell
    d.c0 = 3.0
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, float(np.ceil(pos.max() / cell) * cell + cell)
    eq = pa.define_equation(f"cells_{abs(hash((n, body))) % 10**9}", body)
    with pa.Context(d) as ctx:
        for a, k in enumerate("xyz"):
            ctx.upload(k, np.ascontiguousarray(pos[:, a]))
        ctx.upload("mass", mass)
        ctx.run_equations([eq], pa.LOOP_CELLS, cutoff)
        return ctx.download("s"), ctx.download("c")


BODY = "{ s[i] += mass[j]; c[i] += 1.0 }"


@pytest.mark.parametrize("n,extent", [(1, 3.0), (63, 3.0), (64, 3.0), (65, 4.0), (700, 2.0),      # one cell block: long runs
                                      (2600, 6.0), (5000, 6.0), (64 * 256, 24.0), (64 * 300 + 5, 24.0)])
@pytest.mark.parametrize("precision", [pa.F64, pa.F32])
def test_every_neighbour_once(n, extent, precision):
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, extent, (n, 3)).astype(np.float32).astype(np.float64)
    mass = rng.integers(1, 9, n).astype(np.float64)
    s, c = _run(pos, mass, 2.0, 1.7, BODY, precision)
    near = cKDTree(pos).query_ball_point(pos, 1.7)
    assert np.array_equal(c, [len(v) for v in near])
    assert np.array_equal(s, [mass[v].sum() for v in near])


def test_constants_keep_their_values_in_pair_bodies():
    rng = np.random.default_rng(0)
    pos = rng.uniform(0.0, 2.0, (600, 3))     # runs of 600 candidates: several scans of 128
    s, c = _run(pos, np.ones(600), 2.0, 1.7, "{ s[i] += c0 * mass[j]; c[i] += 1.0 }")
    assert np.array_equal(s, 3.0 * c)
