"""eq1 over the cell iterator with cutoffs far below the cell size, down to where
offsets counted in cutoffs leave FP32's range: every force is the oracle's bit for
bit, in a context and without allocating."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import prestige_amd as pa
from helpers import oracle_state, upload_all
from test_zz_no_alloc import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 4, 4), (6, 5, 4)])   # in the first the cell after a row is a neighbour
@pytest.mark.parametrize("cutoff", [1e-3, 1e-10, 1e-15, 1e-18, 3e-20, 1e-25, 1e-40, 1e-170, 1e-310])
def test_forces_match_the_oracle(cutoff, dims):
    rng = np.random.default_rng(11)
    n = 1003   # the last wavefront and most rows of candidates end within a batch
    pts = rng.uniform(0.0, 1.0, (n, 3)) * dims
    pts[1::9] = pts[0:-1:9]            # coincident pairs
    pts[2::9] = pts[0:-2:9]
    pts[2::9, 0] += 0.25 * cutoff      # and, where FP64 can tell, pairs just inside
    pts = np.minimum(pts, np.asarray(dims) * (1.0 - 1e-9))
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.cell_size = 1.0
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, float(dims[a])
    arrs = {k: np.ascontiguousarray(pts[:, a]) for a, k in enumerate("xyz")}
    force0, mass = rng.standard_normal(n), rng.random(n)
    st = oracle_state(d, {**arrs, "vx": np.zeros(n), "vy": np.zeros(n), "vz": np.zeros(n)})
    assert st.build() == 0
    expect = st.eq1_cells(cutoff, force0, mass)
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        ctx.upload("force", force0)
        ctx.upload("mass", mass)
        ctx.eval_equation(pa.EQ1, pa.LOOP_CELLS, cutoff)
        assert np.array_equal(ctx.download("force"), expect)
    dev = [DeviceArray(v) for v in (arrs["x"], arrs["y"], arrs["z"], mass, force0)]
    lo, hi = (C.c_double * 3)(0, 0, 0), (C.c_double * 3)(*map(float, dims))
    assert pa.load_library().prestige_eq1_cells_noalloc(*[v.p for v in dev], n, lo, hi, 1.0, cutoff, None) == 0
    got = dev[4].get()
    for v in dev:
        v.free()
    assert np.array_equal(got, expect)
