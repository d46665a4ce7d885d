"""The counting sort of a first build against the radix sort: the same keys,
permutation, ids, cell table and state, in one cell and many, at the edges of a
tile of cells, and from a slot order that is not the ids'."""
from __future__ import annotations

import numpy as np
import pytest

import prestige_amd as pa

pytestmark = pytest.mark.gpu


def _builds(d, states, policy, monkeypatch):
    monkeypatch.setenv("PRESTIGE_SORT", policy)
    out = []
    with pa.Context(d) as ctx:
        for st in states:
            for k, v in st.items():
                ctx.upload(k, v)
            ctx.neighbors_build()
            out.append(ctx.neighbors_download())
            out[-1].update({k: ctx.download(k) for k in st})
    return out


@pytest.mark.parametrize("precision", [pa.F64, pa.F32])
@pytest.mark.parametrize("dims,n", [((1, 1, 1), 1), ((1, 1, 1), 700), ((2, 1, 1), 4096), ((2, 1, 1), 4097), ((3, 2, 1), 257), ((11, 31, 3), 256), ((32, 32, 1), 5000),
                                    ((41, 25, 1), 5000), ((60, 50, 40), 200000), ((300, 300, 1), 64),
                                    ((170, 160, 160), 1000)])   # the last grid and the fuller one of two cells
                                                          # are past the counting sort's limits
def test_same_build_as_the_radix_sort(dims, n, precision, monkeypatch):
    rng = np.random.default_rng(n)
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.precision = precision
    d.cell_size = 1.0
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, float(dims[a])
    states = []
    for crowd in (0.0, 0.5):   # then half of them in one cell, from the order the first build left
        pos = rng.uniform(0.0, 1.0, (n, 3)) * dims * 0.999
        pos[: int(crowd * n)] = rng.uniform(0.0, 0.5, (int(crowd * n), 3))
        states.append({k: np.ascontiguousarray(pos[:, a].astype(np.float32).astype(np.float64)) for a, k in enumerate("xyz")})
    got, want = _builds(d, states, "counting", monkeypatch), _builds(d, states, "radix", monkeypatch)
    for g, w in zip(got, want):
        assert g.keys() == w.keys()
        for k in g:
            assert np.array_equal(g[k], w[k]), k
