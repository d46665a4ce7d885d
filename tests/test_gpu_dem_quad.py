"""The DEM contact pass where its tiles and contact lists can go wrong: partial
16-sphere tiles, and a sphere with as many contacts as a context can hold."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, oracle_state, upload_all

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "wx", "wy", "wz", "ax", "ay", "az")


def _check(d, arrs, steps):
    st = oracle_state(d, arrs)
    assert st.step(steps) == 0
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        ctx.step(steps)
        for k in FIELDS:
            got, ref = ctx.download(k), st.get(k)
            bad = np.flatnonzero(got != ref)
            assert bad.size == 0, f"{k}: {bad.size} values differ, first at {bad[:3]}"
    return st.contact_count()


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 65, 1000])
def test_partial_tiles(n):
    d, arrs = make_scene(pa.SCENE_DEM_POUR, n_target=n, seed=4)
    for k in "xy":
        arrs[k][:] = 0.15 + 0.85 * (arrs[k] - 0.15)
    arrs["z"][:] = 0.85 * (arrs["z"] - arrs["z"].min()) + 0.008
    contacts = _check(d, arrs, 40)
    assert n < 1000 or contacts > 500


@pytest.mark.parametrize("contacts", [5, 31, 32])
def test_contact_list_up_to_its_capacity(contacts):
    """One large sphere touched by small ones all around it, at rest on nothing."""
    d, _ = make_scene(pa.SCENE_DEM_POUR, n_target=4, seed=0)
    R, r = 0.05, 0.006
    k = np.arange(contacts) + 0.5
    th, ph = np.pi * (1 + 5 ** 0.5) * k, np.arccos(1 - 2 * k / contacts)
    dirs = np.stack([np.cos(th) * np.sin(ph), np.sin(th) * np.sin(ph), np.cos(ph)], 1)
    pts = np.concatenate([[[0.15, 0.15, 0.15]], 0.15 + dirs * (R + r) * 0.999])
    n = len(pts)
    d.n_particles = d.n_moving = n
    d.max_contacts = 32
    d.cell_size = 2 * R
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a], d.wall_lo[a], d.wall_hi[a] = 0.0, 0.3, 0.0, 0.3
    rng = np.random.default_rng(contacts)
    arrs = {c: np.ascontiguousarray(pts[:, a]) for a, c in enumerate("xyz")}
    arrs.update({c: rng.uniform(-0.2, 0.2, n) for c in ("vx", "vy", "vz")})
    arrs["radius"] = np.full(n, r)
    arrs["radius"][0] = R
    arrs["mass"] = 2500.0 * 4.0 / 3.0 * np.pi * arrs["radius"] ** 3
    assert _check(d, arrs, 3) >= 2 * contacts - 4
