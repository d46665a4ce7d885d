"""eq1 over the cell iterator where its FP32 decision can go wrong: pairs exactly
at the cutoff, pairs a few units in the last place on either side of it, and
wavefronts whose candidates span more than the stage or far from the origin.
Every force is the oracle's bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import oracle_state, upload_all

pytestmark = pytest.mark.gpu


def _lattice(rng):
    """Unit lattice, cutoff exactly two spacings: six pairs per point lie on it."""
    g = np.stack(np.meshgrid(*[np.arange(12.0)] * 3, indexing="ij"), -1).reshape(-1, 3) + 0.5
    return g, 2.0, 2.0


def _ulps(rng):
    """Pairs at the cutoff times 1 + k 2^-52, k in -3..3, in random directions."""
    c = rng.uniform(3.0, 37.0, (400, 3))
    v = rng.standard_normal((400, 3))
    v /= np.linalg.norm(v, axis=1)[:, None]
    k = rng.integers(-3, 4, 400)[:, None]
    return np.concatenate([c, c + v * 1.7 * (1.0 + k * 2.0 ** -52)]), 2.0, 1.7


def _far(rng):
    """A cluster 10^5 cells from the grid's origin along x."""
    p = rng.uniform(0.0, 6.0, (700, 3))
    p[:, 0] += 2.0e5
    return p, 2.0, 1.9


def _crowded(rng):
    """2,600 points in a 3 x 3 x 3 block of cells: rows of about 290 candidates, wider than the stage."""
    return rng.uniform(0.0, 6.0, (2600, 3)), 2.0, 1.3


@pytest.mark.parametrize("precision", [pa.F64, pa.F32])
@pytest.mark.parametrize("points", [_lattice, _ulps, _far, _crowded])
def test_forces_match_the_oracle(points, precision):
    rng = np.random.default_rng(5)
    pts, cell, cutoff = points(rng)
    if precision == pa.F32:
        pts = pts.astype(np.float32).astype(np.float64)
    n = len(pts)
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.precision = precision
    d.n_particles = d.n_moving = n
    d.cell_size = cell
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, float(np.ceil(pts[:, a].max()) + cell)
    arrs = {k: np.ascontiguousarray(pts[:, a]) for a, k in enumerate("xyz")}
    force0, mass = rng.standard_normal(n), rng.random(n)
    force0[::7] = -0.0
    st = oracle_state(d, {**arrs, "vx": np.zeros(n), "vy": np.zeros(n), "vz": np.zeros(n)})
    assert st.build() == 0
    expect = st.eq1_cells(cutoff, force0, mass)
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        ctx.upload("force", force0)
        ctx.upload("mass", mass)
        ctx.eval_equation(pa.EQ1, pa.LOOP_CELLS, cutoff)
        got = ctx.download("force")
    assert np.array_equal(got, expect)
