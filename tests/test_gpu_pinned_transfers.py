"""Fields to and from the caller's own pinned memory and ordinary memory, around the
sizes at which the way changes: the values arrive whole and nothing beside them is
written; pinned memory takes no longer than the link."""
from __future__ import annotations

import ctypes as C
import time

import numpy as np
import pytest

import prestige_amd as pa
from test_zz_no_alloc import hip

pytestmark = pytest.mark.gpu

DP = C.POINTER(C.c_double)


class Pinned:
    """n doubles of pinned memory as .a."""

    def __init__(self, n):
        self.p = C.c_void_p()
        assert hip().hipHostMalloc(C.byref(self.p), C.c_size_t(8 * n), 0) == 0
        self.a = np.frombuffer((C.c_double * n).from_address(self.p.value), np.float64)

    def free(self):
        assert hip().hipHostFree(self.p) == 0


def _context(n):
    d = pa.desc_init(pa.MODEL_PAIRS)
    d.n_particles = d.n_moving = n
    d.cell_size = 1.0
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, 10.0
    return pa.Context(d)


def _ptr(a):
    return C.cast(a.ctypes.data, DP)


# 64 bytes, 976 KiB (also a small context's whole block), 2 MiB, and past the ring's size
@pytest.mark.parametrize("n", [1, 7, 8, 511, 512, 513, 124927, 124928, 124929, 262143, 262144, 262145, 1100003])
def test_values_and_edges(n):
    lib = pa.load_library()
    rng = np.random.default_rng(n)
    block = Pinned(n + 16)
    with _context(n) as ctx:
        for name in ("x", "mass", "anything"):
            for buf in (block.a, np.empty(n + 16)):
                for off in (0, 5):   # inside the allocation, not at a page
                    want = rng.uniform(0.0, 9.0, n)
                    buf[:] = -1.0
                    buf[off:off + n] = want
                    assert lib.prestige_field_upload(ctx._h, name.encode(), _ptr(buf[off:]), n) == 0
                    buf[:] = -2.0
                    assert lib.prestige_field_download(ctx._h, name.encode(), _ptr(buf[off:]), n) == 0
                    assert np.array_equal(buf[off:off + n], want)
                    assert np.all(buf[:off] == -2.0) and np.all(buf[off + n:] == -2.0)
        # a field refused leaves the one before, whatever memory it came from
        block.a[:n] = np.nan
        assert lib.prestige_field_upload(ctx._h, b"x", _ptr(block.a), n) == 5
        assert np.array_equal(ctx.download("x"), _last(ctx, lib, block, n))
    block.free()


def _last(ctx, lib, block, n):
    assert lib.prestige_field_download(ctx._h, b"x", _ptr(block.a), n) == 0
    assert np.all(np.isfinite(block.a[:n]))
    return block.a[:n]


def test_pinned_memory_takes_the_link():
    """4.6 MB into pinned memory: 88 us, of which the copy itself is 85; through the ring it took 185."""
    n = 571000
    lib = pa.load_library()
    block = Pinned(n)
    dev = C.c_void_p()
    assert hip().hipMalloc(C.byref(dev), C.c_size_t(8 * n)) == 0

    def best(fn):
        took = []
        for _ in range(12):
            t = time.perf_counter()
            assert fn() == 0
            took.append(time.perf_counter() - t)
        return min(took)

    with _context(n) as ctx:
        ctx.upload("mass", np.ones(n))
        plain = best(lambda: hip().hipMemcpy(block.p, dev, C.c_size_t(8 * n), 2))
        field = best(lambda: lib.prestige_field_download(ctx._h, b"mass", _ptr(block.a), n))
    assert hip().hipFree(dev) == 0
    block.free()
    assert field < 1.5 * plain


@pytest.mark.parametrize("n", [1, 3, 4095, 4096, 4097])   # checked on the host up to 4,096 values, then on the device
@pytest.mark.parametrize("name,value,status", [("x", np.nan, 5), ("x", -np.inf, 5), ("radius", np.inf, 5), ("radius", 0.0, 1),
                                               ("radius", -0.1, 1), ("radius", 0.6, 1), ("mass", np.nan, 1), ("mass", 0.0, 1)])
def test_one_bad_value(n, name, value, status):
    d = pa.desc_init(pa.MODEL_DEM)
    d.n_particles = d.n_moving = n
    d.cell_size, d.dt = 1.0, 1e-5
    for a in range(3):
        d.grid_lo[a], d.grid_hi[a] = 0.0, 10.0
    good = np.random.default_rng(n).uniform(0.1, 0.5, n)
    good[0] = 0.5   # a radius of half a cell is allowed
    with pa.Context(d) as ctx:
        ctx.upload(name, good)
        for at in {0, n // 2, n - 1}:
            bad = good.copy()
            bad[at] = value
            with pytest.raises(pa.PrestigeError) as e:
                ctx.upload(name, bad)
            assert e.value.status == status
        if name != "mass":   # (the equations' mass is replaced before the check)
            assert np.array_equal(ctx.download(name), good)
        ctx.upload(name, good)
        assert np.array_equal(ctx.download(name), good)
