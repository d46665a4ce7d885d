"""Fields downloaded after an adjoint sweep: rho and p belong to one step, whether
the sweep recomputed segments or not, and a second sweep leaves them as the first."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, upload_all

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [pa.F64, pa.MIXED])
@pytest.mark.parametrize("steps,every", [(4, 4), (6, 2), (7, 3), (5, 1)])
def test_density_and_pressure_are_of_one_step(steps, every, precision):
    d, arrs = make_scene(pa.SCENE_DAM_BREAK, n_target=4000, dx=0.005, precision=precision)
    with pa.Context(d) as ctx:
        upload_all(ctx, {k: arrs[k] for k in ("x", "y", "z", "vx", "vy", "vz")})
        ctx.step(40)   # settle, so that densities differ from step to step
        ctx.forward_tape(steps, every)
        seed = np.ones(3 * ctx.n)
        got = []
        for _ in range(2):
            ctx.adjoint(seed, seed)
            got.append((ctx.download("rho"), ctx.download("p")))
    assert all(np.array_equal(a, b) for a, b in zip(got[0], got[1]))
    rho, p = got[0]
    B = d.rho0 * d.c0 ** 2 / 7.0
    expect = np.maximum(B * ((rho / d.rho0) ** 7 - 1.0), 0.0)
    # rho as downloaded is rounded to 2^-24 in the mixed form, p to as much of itself
    eps = 2.0 ** -24 if precision == pa.MIXED else 2.0 ** -53
    assert np.all(np.abs(p - expect) <= 32 * eps * B + 2 * eps * np.abs(p))
    assert np.any(p > 0.0)
