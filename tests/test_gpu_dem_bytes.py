"""Algorithmic bytes of the DEM contact pass: what it must move for a particle, with
no wall springs, which only spheres at a wall have."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all

pytestmark = pytest.mark.gpu


# gathered position + radius, velocity + mass, angular velocity; id, key; state in and out; next key; the contact
# count and six contacts of a partner id and a spring, in and out
@pytest.mark.parametrize("precision,name,real", [(pa.F64, "dem_force_f64", 8), (pa.MIXED, "dem_force_mixed", 4)])
def test_bytes_of_the_contact_pass(precision, name, real):
    d, arrs = make_scene(pa.SCENE_DEM_POUR, n_target=3000, seed=5, precision=precision)
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        ctx.timing_enable()
        ctx.step(2)
        got = {k["kernel"]: k["bytes_per_launch"] for k in ctx.timing()}
        cells = float(np.prod([int(v) for v in ctx.grid_dims()]))
    per = 11 * real + 4 + 4 + 6 * 32 + 4 + 2 * (4 + 6 * (4 + 3 * real))
    assert got[name] == pytest.approx(per * 3000 + 4 * cells, rel=1e-12)
