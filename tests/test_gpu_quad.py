"""The WCSPH passes with four lanes per particle against the one-lane passes
(the same bits in every form) and the FP64 oracle, at the sizes where they can
go wrong: partial tiles, particles with more neighbours than a list holds, and
tiles whose candidate ranges span thousands of slots."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa
from helpers import make_scene, oracle_state, upload_all

pytestmark = pytest.mark.gpu

FIELDS = ("x", "y", "z", "vx", "vy", "vz", "rho", "p", "ax", "ay", "az")


def _run(d, arrs, steps, mode, monkeypatch):
    monkeypatch.setenv("PRESTIGE_QUAD", mode)
    with pa.Context(d) as ctx:
        upload_all(ctx, arrs)
        ctx.step(steps)
        return {k: ctx.download(k) for k in FIELDS}


def _same(a, b):
    for k in FIELDS:
        bad = np.flatnonzero(a[k] != b[k])
        assert bad.size == 0, f"{k}: {bad.size} values differ, first at {bad[:3]}"


def _stirred(n_target, precision, seed=1):
    d, arrs = make_scene(pa.SCENE_DAM_BREAK, n_target=n_target, dx=0.005, precision=precision)
    rng = np.random.default_rng(seed)
    nf = d.n_moving
    for k in "xyz":
        arrs[k][:nf] += rng.uniform(-5e-4, 5e-4, nf)
    for k in ("vx", "vy", "vz"):
        arrs[k][:nf] = rng.uniform(-0.03, 0.03, nf) * d.c0
    return d, arrs


@pytest.mark.parametrize("n_target", [1, 27, 1000, 8000])
@pytest.mark.parametrize("precision,flags", [(pa.F64, 0), (pa.F32, 0), (pa.MIXED, 0), (pa.MIXED, pa.FLAG_DENSITY_F64)])
def test_same_bits_as_one_lane_per_particle(n_target, precision, flags, monkeypatch):
    d, arrs = _stirred(n_target, precision)
    d.flags = flags
    _same(_run(d, arrs, 25, "on", monkeypatch), _run(d, arrs, 25, "off", monkeypatch))


def _free(points, h, cell, lo, hi):
    """Points as moving particles in an open grid."""
    d, _ = make_scene(pa.SCENE_DAM_BREAK, n_target=8, dx=0.005)
    d.n_particles = d.n_moving = len(points)
    d.h, d.cell_size = h, cell
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = lo[a], hi[a]
    arrs = {k: np.ascontiguousarray(points[:, a]) for a, k in enumerate("xyz")}
    rng = np.random.default_rng(3)
    arrs.update({k: rng.uniform(-0.01, 0.01, len(points)) for k in ("vx", "vy", "vz")})
    return d, arrs


def _crowd():
    """A 12 x 6 x 6 block with two layers per cell pair in y and z: rows of at most 99 candidates, interior
    particles with more than 128 neighbours."""
    s = 0.005
    g = np.stack(np.meshgrid(np.arange(12), np.arange(6), np.arange(6), indexing="ij"), -1).reshape(-1, 3)
    cell = 3.4 * s
    pts = (g + 0.5) * s + np.array([cell, 2 * cell - 3 * s, 2 * cell - 3 * s])
    return _free(pts, 1.7 * s, cell, (0.0, 0.0, 0.0), (8 * cell, 4 * cell, 4 * cell))


def _plate():
    """Two far corners in one cell layer under a full layer of 6,400 particles: the corners share a tile, and
    their rows in the layer above span all of it."""
    s = 0.005
    cell = 2.4 * s
    g = np.stack(np.meshgrid(np.arange(80), np.arange(80), indexing="ij"), -1).reshape(-1, 2)
    top = np.column_stack([(g + 0.5) * s, np.full(len(g), 1.1 * cell)])
    corners = np.array([[0.4 * s, 0.4 * s, 0.9 * cell], [79.4 * s, 79.4 * s, 0.9 * cell]])
    return _free(np.concatenate([corners, top]), 1.2 * s, cell, (0.0, 0.0, 0.0), (80 * s, 80 * s, 3 * cell))


@pytest.mark.parametrize("scene", [_crowd, _plate])
def test_lists_that_do_not_fit(scene, monkeypatch):
    d, arrs = scene()
    if scene is _crowd:
        P = np.stack([arrs[k] for k in "xyz"], 1)
        nb = (((P[:, None] - P[None]) ** 2).sum(2) < (2 * d.h) ** 2).sum(1)
        assert nb.max() > 128
    st = oracle_state(d, arrs)
    assert st.step(2) == 0
    got = _run(d, arrs, 2, "on", monkeypatch)
    _same(got, {k: st.get(k) for k in FIELDS})
    for precision in (pa.F32, pa.MIXED):
        d.precision = precision
        _same(_run(d, arrs, 2, "on", monkeypatch), _run(d, arrs, 2, "off", monkeypatch))


@pytest.mark.parametrize("precision", [pa.F64, pa.MIXED])
@pytest.mark.parametrize("n_target", [27, 8000])
def test_adjoint_same_bits(n_target, precision, monkeypatch):
    """Steps recorded by the four-lane passes and reverse passes split over a block's wavefronts give the
    gradients of the one-lane, one-wavefront passes bit for bit."""
    d, arrs = _stirred(n_target, precision)
    rng = np.random.default_rng(2)
    seeds = [rng.standard_normal((3, d.n_particles)) for _ in range(2)]
    out = {}
    for mode in ("on", "off"):
        monkeypatch.setenv("PRESTIGE_QUAD", mode)
        with pa.Context(d) as ctx:
            upload_all(ctx, arrs)
            ctx.forward_tape(14, 4)
            out[mode] = ctx.adjoint(*seeds)
    assert np.array_equal(out["on"][0], out["off"][0])
    assert np.array_equal(out["on"][1], out["off"][1])
