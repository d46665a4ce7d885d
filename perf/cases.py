"""The work a program has this library do, as measurable cases.

listed() names twelve of them and draw() gives more of the same ranges.  Every
simulation case is one self-contained run, as a parameter study or a
calibration loop makes it: the initial state goes up, the steps run, the final
state comes back.  The context (grid, constants, device buffers) is what such a
program keeps between runs, so prepare() makes it.

exact() restates each case's mathematics in float64 torch: neighbour pairs from
a sorted cell list, plain index_add sums, automatic differentiation for the
adjoints.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

import prestige_amd as pa

FORMS = {"f64": pa.F64, "f32": pa.F32, "mixed": pa.MIXED}
STATE = ("x", "y", "z", "vx", "vy", "vz")
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # A tank of 8,000 fluid particles (42,866 with its walls): the size of a first experiment,
        # where a step is a handful of short launches.
        {"name": "wcsph_f64_8k", "kind": "wcsph", "form": "f64", "fluid": 8000, "steps": 100},
        # A tank for interactive or batch studies in the mixed form, 64,000 fluid particles.
        {"name": "wcsph_mixed_64k", "kind": "wcsph", "form": "mixed", "fluid": 64000, "steps": 100},
        # An odd size (67^3) in single precision.
        {"name": "wcsph_f32_300k", "kind": "wcsph", "form": "f32", "fluid": 300763, "steps": 100},
        # The million-particle dam break in the mixed form.
        {"name": "wcsph_mixed_1M", "kind": "wcsph", "form": "mixed", "fluid": 1000000, "steps": 100},
        # The largest workload of the benchmark: 4,019,679 fluid particles in FP64.
        {"name": "wcsph_f64_4M", "kind": "wcsph", "form": "f64", "fluid": 4000000, "steps": 100},
        # 10,000 equal spheres, a lightly compressed bed: the smallest granular workload of the benchmark.
        {"name": "dem_lattice_f64_10k", "kind": "dem", "form": "f64", "scene": "lattice", "spheres": 10000, "steps": 100},
        # 100,000 polydisperse spheres colliding in a bin, mixed form.
        {"name": "dem_pour_mixed_100k", "kind": "dem", "form": "mixed", "scene": "pour", "spheres": 100000, "steps": 100},
        # Gradients of a dam break with respect to (alpha, c0) and the initial velocities.
        {"name": "adjoint_wcsph_mixed_27k", "kind": "adjoint_wcsph", "form": "mixed", "fluid": 27000, "steps": 20, "every": 5},
        # Gradients of a granular run with respect to (kn, e, mu) and the initial velocities.
        {"name": "adjoint_dem_f64_20k", "kind": "adjoint_dem", "form": "f64", "scene": "pour", "spheres": 20000, "steps": 60,
         "every": 15},
        # The reference's own loop, force[i] += mass[j] over all pairs, at its benchmark size.
        {"name": "eq1_allpairs_10k", "kind": "allpairs", "n": 10000},
        # The same equation over the cell iterator on the caller's device arrays: keys, sort, cell table, gather.
        {"name": "eq1_cells_1M", "kind": "cells", "n": 1000000, "cutoff": 2.4},
        # The density and state equations as generated kernels on new positions.
        {"name": "generated_density_250k", "kind": "generated", "fluid": 250047},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["wcsph", "wcsph", "wcsph", "dem", "dem", "adjoint_wcsph", "adjoint_dem", "allpairs", "cells", "generated"])
    if kind == "wcsph":
        return {"kind": kind, "form": rng.choice(["f64", "f32", "mixed"]), "fluid": _log_int(rng, 1000, 2500000),
                "steps": rng.randrange(20, 81)}
    if kind == "dem":
        scene = rng.choice(["lattice", "pour"])
        return {"kind": kind, "form": rng.choice(["f64", "mixed"]), "scene": scene,
                "spheres": _log_int(rng, 500, 12000 if scene == "lattice" else 400000), "steps": rng.randrange(20, 101)}
    if kind == "adjoint_wcsph":
        steps = rng.randrange(6, 31)
        return {"kind": kind, "form": rng.choice(["f64", "mixed"]), "fluid": _log_int(rng, 1000, 200000), "steps": steps,
                "every": rng.randrange(2, steps + 1)}
    if kind == "adjoint_dem":
        steps = rng.randrange(10, 81)
        return {"kind": kind, "form": rng.choice(["f64", "mixed"]), "scene": "pour", "spheres": _log_int(rng, 500, 100000),
                "steps": steps, "every": rng.randrange(3, steps + 1)}
    if kind == "allpairs":
        return {"kind": kind, "n": _log_int(rng, 300, 60000)}
    if kind == "cells":
        return {"kind": kind, "n": _log_int(rng, 1000, 1048576), "cutoff": round(rng.uniform(1.6, 2.6), 2)}
    return {"kind": kind, "fluid": _log_int(rng, 1000, 1000000)}


# -- inputs ----------------------------------------------------------------------
def _dam(case, seed):
    """A dam break part-way into its motion: fluid off its lattice sites and moving at up to a few percent of c0."""
    d, a = pa.scene(pa.SCENE_DAM_BREAK, n_target=case["fluid"], dx=0.005)
    rng = np.random.default_rng(seed)
    nf = int(d.n_moving)
    for k in ("x", "y", "z"):
        a[k][:nf] += rng.uniform(-0.1, 0.1, nf) * 0.005
    for k in ("vx", "vy", "vz"):
        a[k][:nf] = rng.uniform(-0.03, 0.03, nf) * d.c0
    return d, a


def _bed(case, seed):
    """Spheres in contact: the scene's lattice drawn together to a lightly compressed bed on the floor."""
    lattice = case["scene"] == "lattice"
    d, a = pa.scene(pa.SCENE_DEM_LATTICE if lattice else pa.SCENE_DEM_POUR, n_target=case["spheres"], seed=seed % (1 << 63))
    f = 0.95 if lattice else 0.85
    for ax, k in enumerate(("x", "y")):
        mid = 0.5 * (d.wall_lo[ax] + d.wall_hi[ax])
        a[k][:] = mid + f * (a[k] - mid)
    low = float((a["z"] - a["radius"]).min())
    a["z"][:] = f * (a["z"] - low) - 0.0002 + (1.0 - f) * 0.01
    return d, a


def _ctx(d, case):
    d.precision = FORMS[case["form"]]
    return pa.Context(d)


def prepare(case, seed):
    kind = case["kind"]
    rng = np.random.default_rng(seed + 1)
    if kind in ("wcsph", "adjoint_wcsph"):
        d, a = _dam(case, seed)
    elif kind in ("dem", "adjoint_dem"):
        d, a = _bed(case, seed)
    if kind in ("wcsph", "dem"):
        return {"case": case, "ctx": _ctx(d, case), "arrays": a}
    if kind in ("adjoint_wcsph", "adjoint_dem"):
        n = int(d.n_particles)
        seeds = [rng.standard_normal((3, n)) for _ in range(2)]
        return {"case": case, "ctx": _ctx(d, case), "arrays": a, "seeds": seeds}
    if kind == "allpairs":
        n = case["n"]
        d = pa.desc_init(pa.MODEL_PAIRS)
        d.n_particles = d.n_moving = n
        d.cell_size = 0.1
        for ax in range(3):
            d.grid_lo[ax], d.grid_hi[ax] = 0.0, 1.0
        ctx = pa.Context(d)
        ctx.upload("mass", rng.uniform(0.5, 1.5, n))
        return {"case": case, "ctx": ctx, "force": rng.standard_normal(n)}
    if kind == "cells":
        x, y, z, mass, force, hi = _box(case, seed)
        dev = [torch.from_numpy(v).to(DEV) for v in (x, y, z, mass, force)]
        cs = float(case["cutoff"])
        return {"case": case, "dev": dev, "lo": (C.c_double * 3)(0.0, 0.0, 0.0), "hi": (C.c_double * 3)(hi, hi, hi), "cs": cs}
    d, a = _dam(case, seed)
    d.model = pa.MODEL_PAIRS
    ctx = pa.Context(d)
    ctx.upload("mass", np.full(int(d.n_particles), d.mass))
    return {"case": case, "ctx": ctx, "arrays": a, "zero": np.zeros(int(d.n_particles)), "cutoff": float(d.cell_size)}


def _box(case, seed):
    """n points about one apart in a cube, in no particular order."""
    n = case["n"]
    rng = np.random.default_rng(seed)
    side = math.ceil(n ** (1.0 / 3.0) - 1e-9)
    sites = rng.permutation(side ** 3)[:n]
    p = [(sites % side) + rng.uniform(0.05, 0.95, n), (sites // side % side) + rng.uniform(0.05, 0.95, n),
         (sites // (side * side)) + rng.uniform(0.05, 0.95, n)]
    return (*p, rng.uniform(0.5, 1.5, n), rng.standard_normal(n), float(side))


# -- one pass ---------------------------------------------------------------------
def _upload(s):
    ctx, a = s["ctx"], s["arrays"]
    for k in STATE:
        ctx.upload(k, a[k])
    if "radius" in a:
        ctx.upload("radius", a["radius"])
        ctx.upload("mass", a["mass"])
        zero = s.setdefault("zero", np.zeros_like(a["x"]))
        for k in ("wx", "wy", "wz"):   # spin starts again from rest
            ctx.upload(k, zero)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("wcsph", "dem"):
        _upload(s)
        s["ctx"].step(case["steps"])
        return {k: s["ctx"].download(k) for k in STATE + (("rho",) if kind == "wcsph" else ("wx", "wy", "wz"))}
    if kind in ("adjoint_wcsph", "adjoint_dem"):
        _upload(s)
        s["ctx"].forward_tape(case["steps"], case["every"])
        gp, gv = s["ctx"].adjoint(*s["seeds"])
        return {"params": gp, "v0": gv}
    if kind == "allpairs":
        s["ctx"].upload("force", s["force"])
        s["ctx"].eval_equation(pa.EQ1, pa.LOOP_ALLPAIRS)
        return s["ctx"].download("force")
    if kind == "cells":
        x, y, z, mass, force = s["dev"]
        out = force.clone()
        status = pa.load_library().prestige_eq1_cells_noalloc(
            x.data_ptr(), y.data_ptr(), z.data_ptr(), mass.data_ptr(), out.data_ptr(), x.numel(), s["lo"], s["hi"], s["cs"],
            s["cs"], C.c_void_p(torch.cuda.current_stream().cuda_stream))
        if status:
            raise RuntimeError(f"prestige_eq1_cells_noalloc: status {status}")
        return out
    ctx, a = s["ctx"], s["arrays"]
    for k in ("x", "y", "z"):
        ctx.upload(k, a[k])
    ctx.upload("rho", s["zero"])
    ctx.run_equations([pa.EQ_SPH_DENSITY, pa.EQ_SPH_EOS], pa.LOOP_CELLS, s["cutoff"])
    return {k: ctx.download(k) for k in ("rho", "p")}


# -- what one pass cannot do without ------------------------------------------------
def _dam_counts(fluid):
    side = math.ceil(fluid ** (1.0 / 3.0) - 1e-9)
    ix, iy, iz = round(3.2 * side), round(1.34 * side), round(2.4 * side)
    nf = side ** 3
    return nf, nf + (ix + 6) * (iy + 6) * (iz + 3) - ix * iy * iz


def work(case):
    kind = case["kind"]
    if kind in ("wcsph", "adjoint_wcsph"):
        nf, n = _dam_counts(case["fluid"])
        scalar = 4.0 if case["form"] == "f32" else 8.0
        # per step: density reads positions and writes rho; force reads the state and rho, writes the state;
        # 57 neighbours each, about 15 and 45 operations a pair
        step = {"bytes": n * 4 * scalar + nf * 13 * scalar, "flops": 57.0 * (15.0 * n + 45.0 * nf)}
        if kind == "wcsph":
            return {k: v * case["steps"] + (13 * 8.0 * n if k == "bytes" else 0.0) for k, v in step.items()}
        # forward and reverse sweep, the reverse pair bodies about 2.5 times the forward ones
        return {k: v * case["steps"] * 3.5 + (15 * 8.0 * n if k == "bytes" else 0.0) for k, v in step.items()}
    if kind in ("dem", "adjoint_dem"):
        n = case["spheres"]
        # per step: state in and out (9 + r + m), contact history of about 4 contacts in and out; 120 operations a contact
        step = {"bytes": n * (8.0 * 20 + 2 * 4 * 28.0), "flops": n * 4 * 120.0}
        if kind == "dem":
            return {k: v * case["steps"] + (20 * 8.0 * n if k == "bytes" else 0.0) for k, v in step.items()}
        return {k: v * case["steps"] * 3.5 + (20 * 8.0 * n if k == "bytes" else 0.0) for k, v in step.items()}
    if kind == "allpairs":
        return {"bytes": 24.0 * case["n"], "flops": float(case["n"]) ** 2}
    if kind == "cells":
        near = 4.0 / 3.0 * math.pi * case["cutoff"] ** 3
        return {"bytes": 48.0 * case["n"], "flops": case["n"] * near * 9.0}
    _, n = _dam_counts(case["fluid"])
    return {"bytes": 56.0 * n, "flops": 57.0 * 15.0 * n}


# -- the same mathematics in float64 torch -------------------------------------------
def _pairs(pos, lo, cs, dims, reach):
    """Ordered pairs (i, j), j == i left out, with |x_i - x_j| < reach[i, j]; reach(i, j) gives the distance."""
    n = pos.shape[0]
    nx, ny, nz = dims
    cell = torch.floor((pos - lo) / cs).long()
    key = (cell[:, 2] * ny + cell[:, 1]) * nx + cell[:, 0]
    skey, order = torch.sort(key, stable=True)
    start = torch.searchsorted(skey, torch.arange(nx * ny * nz + 1, device=pos.device))
    x0, x1 = (cell[:, 0] - 1).clamp(min=0), (cell[:, 0] + 1).clamp(max=nx - 1)
    me = torch.arange(n, device=pos.device)
    out_i, out_j = [], []
    for dz in (-1, 0, 1):
        for dy in (-1, 0, 1):
            z, y = cell[:, 2] + dz, cell[:, 1] + dy
            ok = (z >= 0) & (z < nz) & (y >= 0) & (y < ny)
            row = (z.clamp(0, nz - 1) * ny + y.clamp(0, ny - 1)) * nx
            j0 = start[row + x0]
            cnt = torch.where(ok, start[row + x1 + 1] - j0, torch.zeros_like(j0))
            i = torch.repeat_interleave(me, cnt)
            first = torch.cumsum(cnt, 0) - cnt
            j = order[j0[i] + torch.arange(i.numel(), device=pos.device) - first[i]]
            keep = (i != j) & (((pos[i] - pos[j]) ** 2).sum(1) < reach(i, j) ** 2)
            out_i.append(i[keep])
            out_j.append(j[keep])
    return torch.cat(out_i), torch.cat(out_j)


def _grid(d):
    dims = [int(math.ceil((d.grid_hi[a] - d.grid_lo[a]) / d.cell_size)) for a in range(3)]
    return torch.tensor(list(d.grid_lo), dtype=torch.float64, device=DEV), float(d.cell_size), dims


def _spline(q):
    return torch.where(q < 1.0, 1.0 + q * q * (0.75 * q - 1.5), 0.25 * (2.0 - q).clamp(min=0.0) ** 3)


def _density(pos, i, j, d):
    q = (pos[i] - pos[j]).norm(dim=1) / d.h
    sigma = 1.0 / (math.pi * d.h ** 3)
    one = torch.ones(pos.shape[0], dtype=torch.float64, device=pos.device)
    return d.mass * sigma * one.index_add(0, i, _spline(q))


def _sph(case, seed, grads):
    d, a = _dam(case, seed)
    pos = torch.tensor(np.stack([a[k] for k in STATE[:3]], 1), device=DEV)
    v0 = torch.tensor(np.stack([a[k] for k in STATE[3:]], 1), device=DEV)
    n, nf = pos.shape[0], int(d.n_moving)
    lo, cs, dims = _grid(d)
    alpha, c0 = (torch.tensor(v, dtype=torch.float64, device=DEV) for v in (d.alpha, d.c0))
    if grads:
        for t in (v0, alpha, c0):
            t.requires_grad_(True)
    gvec = torch.tensor(list(d.gravity), dtype=torch.float64, device=DEV)
    moves = (torch.arange(n, device=DEV) < nf)[:, None]
    vel, rho, sigma = v0, None, 1.0 / (math.pi * d.h ** 3)
    for _ in range(case["steps"]):
        with torch.no_grad():
            i, j = _pairs(pos, lo, cs, dims, lambda i, j: 2.0 * d.h)
        rho = _density(pos, i, j, d)
        p = ((d.rho0 * c0 * c0 / 7.0) * ((rho / d.rho0) ** 7 - 1.0)).clamp(min=0.0)
        pr = p / (rho * rho)
        keep = i < nf   # only moving particles feel a force
        i, j = i[keep], j[keep]
        dx, dv = pos[i] - pos[j], vel[i] - vel[j]
        r2 = (dx * dx).sum(1)
        r = r2.sqrt()
        q = r / d.h
        df = torch.where(q < 1.0, q * (2.25 * q - 3.0), -0.75 * (2.0 - q).clamp(min=0.0) ** 2)
        w = (dx * dv).sum(1)
        mu = d.h * w / (r2 + 0.01 * d.h * d.h)
        visc = torch.where(w < 0.0, -alpha * c0 * mu / (0.5 * (rho[i] + rho[j])), torch.zeros_like(w))
        s = (pr[i] + pr[j] + visc) * df / r
        acc = torch.zeros_like(pos).index_add(0, i, s[:, None] * dx)
        acc = gvec - (d.mass * sigma / d.h) * acc
        vel = torch.where(moves, vel + d.dt * acc, vel)
        pos = torch.where(moves, pos + d.dt * vel, pos)
    return pos, vel, rho, (alpha, c0), v0, nf


def _tangential(fn, nrm, vt, xi, kt, mu, dt):
    xi = xi - (xi * nrm).sum(-1, keepdim=True) * nrm + vt * dt
    ft = -kt * xi
    f2 = (ft * ft).sum(-1, keepdim=True)
    ftn = torch.where(f2 > 0.0, f2, torch.ones_like(f2)).sqrt() * (f2 > 0.0)
    cap = mu * fn.abs()[..., None]
    slip = ftn > cap
    ft = torch.where(slip, ft * (cap / torch.where(slip, ftn, torch.ones_like(ftn))), ft)
    return ft, torch.where(slip, -ft / kt, xi)


def _dem(case, seed, grads):
    d, a = _bed(case, seed)
    pos, v0 = (torch.tensor(np.stack([a[k] for k in ks], 1), device=DEV) for ks in (STATE[:3], STATE[3:]))
    rad, mass = (torch.tensor(a[k], device=DEV) for k in ("radius", "mass"))
    n = pos.shape[0]
    lo, cs, dims = _grid(d)
    kn, e, mu = (torch.tensor(v, dtype=torch.float64, device=DEV) for v in (d.kn, d.restitution, d.mu))
    if grads:
        for t in (kn, e, mu, v0):
            t.requires_grad_(True)
    kt = kn * (d.kt / d.kn)
    le = torch.log(e)
    two_zeta = -2.0 * le / torch.sqrt(math.pi ** 2 + le * le)
    gvec = torch.tensor(list(d.gravity), dtype=torch.float64, device=DEV)
    vel, om = v0, torch.zeros_like(v0)
    old_key = torch.empty(0, dtype=torch.long, device=DEV)
    old_xi = torch.zeros((0, 3), dtype=torch.float64, device=DEV)
    wxi = {w: torch.zeros_like(pos) for w in range(6)}
    for _ in range(case["steps"]):
        with torch.no_grad():
            i, j = _pairs(pos, lo, cs, dims, lambda i, j: rad[i] + rad[j])
            key, order = torch.sort(i * n + j)
            i, j = i[order], j[order]
            at = torch.searchsorted(old_key, key).clamp(max=max(0, old_key.numel() - 1))
            had = (old_key[at] == key) if old_key.numel() else torch.zeros_like(key, dtype=torch.bool)
        xi = torch.where(had[:, None], old_xi[at], torch.zeros((1, 3), dtype=torch.float64, device=DEV)) if old_key.numel() \
            else torch.zeros((key.numel(), 3), dtype=torch.float64, device=DEV)
        dx = pos[i] - pos[j]
        dist = dx.norm(dim=1)
        nrm = dx / dist[:, None]
        vr = vel[i] - vel[j] - torch.linalg.cross(rad[i, None] * om[i] + rad[j, None] * om[j], nrm)
        vn = (vr * nrm).sum(1)
        meff = mass[i] * mass[j] / (mass[i] + mass[j])
        fn = kn * (rad[i] + rad[j] - dist) - two_zeta * torch.sqrt(meff * kn) * vn
        ft, xi = _tangential(fn, nrm, vr - vn[:, None] * nrm, xi, kt, mu, d.dt)
        force = torch.zeros_like(pos).index_add(0, i, fn[:, None] * nrm + ft)
        torque = torch.zeros_like(pos).index_add(0, i, -rad[i, None] * torch.linalg.cross(nrm, ft))
        old_key, old_xi = key, xi
        for w in range(6):
            if not d.wall_mask >> w & 1:
                continue
            ax, sg = w >> 1, -1.0 if w & 1 else 1.0
            gap = d.wall_hi[ax] - pos[:, ax] if w & 1 else pos[:, ax] - d.wall_lo[ax]
            delta = rad - gap
            on = (delta.detach() > 0.0)[:, None]
            nrm = torch.zeros_like(pos)
            nrm[:, ax] = sg
            vr = vel - torch.linalg.cross(rad[:, None] * om, nrm)
            vn = (vr * nrm).sum(1)
            fn = kn * delta - two_zeta * torch.sqrt(mass * kn) * vn
            ft, wx = _tangential(fn, nrm, vr - vn[:, None] * nrm, wxi[w], kt, mu, d.dt)
            zero = torch.zeros_like(ft)
            wxi[w] = torch.where(on, wx, zero)
            force = force + torch.where(on, fn[:, None] * nrm + ft, zero)
            torque = torque + torch.where(on, -rad[:, None] * torch.linalg.cross(nrm, ft), zero)
        vel = vel + d.dt * (force / mass[:, None] + gvec)
        pos = pos + d.dt * vel
        om = om + d.dt * torque / (0.4 * mass * rad * rad)[:, None]
    return pos, vel, om, (kn, e, mu), v0, n


def _numpy(t):
    return t.detach().cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    fast = DEV == "cuda"
    if kind in ("wcsph", "adjoint_wcsph"):
        n = _dam_counts(case["fluid"])[1] * case["steps"]
        if n > ((8e7 if kind == "wcsph" else 4e6) if fast else 5e6 if kind == "wcsph" else 4e5):
            return None
        pos, vel, rho, params, v0, nf = _sph(case, seed, kind != "wcsph")
        if kind == "wcsph":
            return {**{k: _numpy(pos[:, c]) for c, k in enumerate(STATE[:3])},
                    **{k: _numpy(vel[:, c]) for c, k in enumerate(STATE[3:])}, "rho": _numpy(rho)}
    elif kind in ("dem", "adjoint_dem"):
        if case["spheres"] * case["steps"] > (2e7 if fast else 1e6):
            return None
        pos, vel, om, params, v0, nf = _dem(case, seed, kind != "dem")
        if kind == "dem":
            return {**{k: _numpy(pos[:, c]) for c, k in enumerate(STATE[:3])},
                    **{k: _numpy(vel[:, c]) for c, k in enumerate(STATE[3:])},
                    **{k: _numpy(om[:, c]) for c, k in enumerate(("wx", "wy", "wz"))}}
    if kind in ("adjoint_wcsph", "adjoint_dem"):
        rng = np.random.default_rng(seed + 1)
        sx, sv = (torch.tensor(rng.standard_normal((3, pos.shape[0])).T.copy(), device=DEV) for _ in range(2))
        g = torch.autograd.grad((sx * pos).sum() + (sv * vel).sum(), (*params, v0))
        gv = g[-1].clone()
        gv[nf:] = 0.0   # fixed particles' velocities are no parameters
        return {"params": np.array([float(v) for v in g[:-1]]), "v0": _numpy(gv.T.contiguous())}
    if kind == "allpairs":
        rng = np.random.default_rng(seed + 1)
        mass = rng.uniform(0.5, 1.5, case["n"])
        return rng.standard_normal(case["n"]) + math.fsum(mass)
    if kind == "cells":
        x, y, z, mass, force, hi = _box(case, seed)
        pos = torch.tensor(np.stack([x, y, z], 1), device=DEV)
        cs = float(case["cutoff"])
        i, j = _pairs(pos, torch.zeros(3, dtype=torch.float64, device=DEV), cs, [int(math.ceil(hi / cs))] * 3, lambda i, j: cs)
        m = torch.tensor(mass, device=DEV)
        return _numpy((torch.tensor(force, device=DEV) + m).index_add(0, i, m[j]))
    d, a = _dam(case, seed)
    pos = torch.tensor(np.stack([a[k] for k in STATE[:3]], 1), device=DEV)
    lo, cs, dims = _grid(d)
    i, j = _pairs(pos, lo, cs, dims, lambda i, j: 2.0 * d.h)
    rho = _density(pos, i, j, d)
    p = ((d.rho0 * d.c0 * d.c0 / 7.0) * ((rho / d.rho0) ** 7 - 1.0)).clamp(min=0.0)
    return {"rho": _numpy(rho), "p": _numpy(p)}
