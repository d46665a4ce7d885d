// dem_kernels.hpp — DEM contact gather kernel, templated on the precision form.
//
// Bodies: linear spring-dashpot normal force with cn = 2 zeta sqrt(m_eff kn),
// zeta = -ln e / sqrt(pi^2 + ln^2 e); tangential spring xi (projected onto the
// current tangent plane, advanced by v_t dt, Coulomb-capped |Ft| <= mu |Fn|,
// reset when the contact opens); torque (-r_i n) x Ft; half-space walls with
// m_eff = m (Cundall & Strack 1979).  Loop shape of
// prestige/src/codegen/simple_cpu.rs:7-19 over the 27-cell iterator, j != i,
// gather into [i].  The tangential history of particle i lives at index
// id(i) of SoA slot arrays, so the sort never moves it; each step reads the
// previous buffer and writes the next (double-buffered), which is why a
// gather needs no atomics.
//
// kF64: all FP64 (bit-identical to the host oracle; TU built with
// -ffp-contract=off).  kMixed: pair geometry from FP32 offsets to the FP64
// cell origin (metres), forces and history in FP32, walls' distances and the
// integrator in FP64.
#pragma once
#include "sph_kernels.hpp"

namespace prestige {

template <int F> struct DemForm;
template <> struct DemForm<kF64> { using real = double; using G4 = double4; };
template <> struct DemForm<kMixed> { using real = float; using G4 = float4; };

// Tangential spring update (shared by pair and wall contacts); true when the
// spring is at the Coulomb cap (sliding).
template <class real>
__device__ inline bool dem_tangential(real fn, real nx, real ny, real nz, real vtx, real vty, real vtz,
                                      real xox, real xoy, real xoz, real kt, real mu, real neg_inv_kt,
                                      real dt, real* ft, real* xn) {
  real xdn = xox * nx + xoy * ny + xoz * nz;
  real xpx = xox - xdn * nx, xpy = xoy - xdn * ny, xpz = xoz - xdn * nz;
  real xnx = xpx + vtx * dt, xny = xpy + vty * dt, xnz = xpz + vtz * dt;
  real ftx = -kt * xnx, fty = -kt * xny, ftz = -kt * xnz;
  real ftn = sqrt(ftx * ftx + fty * fty + ftz * ftz);
  real fcap = mu * (fn < real(0.0) ? -fn : fn);
  const bool slip = ftn > fcap;
  if (slip) {
    real sc = fcap / ftn;
    ftx = ftx * sc; fty = fty * sc; ftz = ftz * sc;
    xnx = ftx * neg_inv_kt; xny = fty * neg_inv_kt; xnz = ftz * neg_inv_kt;
  }
  ft[0] = ftx; ft[1] = fty; ft[2] = ftz;
  xn[0] = xnx; xn[1] = xny; xn[2] = xnz;
  return slip;
}

// Contact history by particle id: cnt holds the number of pair contacts in bits
// 0-7 and the walls touched in bits 8-13.  The spring of a wall (wxi) is written
// and read for the walls touched only; every other is zero.  18 zeros a particle
// and step were four fifths of what a pour of 100,000 mixed spheres wrote (90 MB of
// 180 moved in all).  Us a pass without them, and with the FP64 state read only
// where the walls need it (FP32 form: 108 -> 85 registers): pour of 100,000 FP64 38
// -> 36, mixed 35 -> 32; of 400,000 FP64 127 -> 106, mixed 105 -> 86.
struct DemHist {
  const uint32_t* cnt_in; const uint32_t* id_in; const void* xi_in; const void* wxi_in;
  uint32_t* cnt_out; uint32_t* id_out; void* xi_out; void* wxi_out;
};

// Contacts of one particle's list in LDS.  desc.max_contacts is at most 32, so
// a particle with more than the list holds raises the capacity flag.
constexpr uint32_t kDemList = 36;

// Four lanes per particle (a quad), 16 particles per wavefront.  First every
// lane tests candidates sub, sub + 4, ... of each row run, and the touching
// ones go into the particle's list in LDS in run and slot order; then each
// lane evaluates one contact of the list at a time, and every lane of the quad
// adds the four in list order (quad permutes), so the sums keep the oracle's
// order.  A step of a small scene is a chain of dependent reads (key, cell
// table, candidates, contacts, history), and the contact body is long: with
// one lane per particle it ran once for every candidate position at which any
// of 64 particles had a contact.
// Us a pass, one lane per particle / this: FP64 lattice of 500 18 / 11, 10,000
// 26 / 15, pour 20,000 57 / 19, 100,000 82 / 39, 400,000 207 / 129; mixed pour
// 100,000 72 / 35, 400,000 150 / 103 (HIP events, which add about 3).
template <int F>
__global__ __launch_bounds__(64) void k_dem_force(
    uint32_t n, uint64_t n_moving, const typename DemForm<F>::G4* __restrict__ gpos,
    const typename DemForm<F>::G4* __restrict__ gvel, const typename DemForm<F>::G4* __restrict__ gom,
    const uint32_t* __restrict__ ids, const uint32_t* __restrict__ skeys,
    const uint32_t* __restrict__ lb, Grid g, DemConst kc, const double4* __restrict__ spos,
    const double4* __restrict__ svel, const double4* __restrict__ som, double4* __restrict__ opos,
    double4* __restrict__ ovel, double4* __restrict__ oom, uint32_t* __restrict__ okeys,
    double4* __restrict__ oforce, DemHist hist, MovedOut moved, uint32_t* flags,
    uint32_t* __restrict__ events, uint32_t ev_weight, uint32_t n_tiles) {
  using real = typename DemForm<F>::real;
  using G4 = typename DemForm<F>::G4;
  __shared__ uint32_t s_list[kQuadSlots][kDemList];
  __shared__ uint32_t s_hid[kQuadSlots][33];   // partner ids of the previous step's contacts
  const uint32_t tile = xcd_tile(blockIdx.x);
  if (tile >= n_tiles) return;
  const uint32_t lane = threadIdx.x, sub = lane & 3u, p = lane >> 2, qshift = lane & ~3u;
  const uint32_t below = (1u << sub) - 1u;
  const uint32_t wbase = tile * kQuadSlots, i = wbase + p;
  const bool in = i < n;
  const uint32_t self = in ? i : wbase;   // a slot every lane may read
  const uint32_t me = ids[self];
  const bool live = in && (uint64_t)me < n_moving;
  const uint32_t mc = kc.max_contacts;
  const real* xi_in = (const real*)hist.xi_in;
  const real* wxi_in = (const real*)hist.wxi_in;
  real* xi_out = (real*)hist.xi_out;
  real* wxi_out = (real*)hist.wxi_out;
  const uint32_t key_i = skeys[self];
  if (in && !live) {   // fixed: the state copies through, without contacts
    if (sub == 0u) {
      opos[i] = spos[i]; ovel[i] = svel[i]; oom[i] = som[i]; okeys[i] = key_i;
      if (oforce) oforce[i] = make_double4(0, 0, 0, 0);
      hist.cnt_out[me] = 0;
    }
  }
  bool mv = false;
  if (__ballot(live) != 0ull) {
    const CellRows cr = decode_cell(key_i, g);
    const G4 pi = gpos[self], vi = gvel[self], wi = gom[self];
    // radius / mass: FP64 form keeps them in pos.w / vel.w; mixed in om.w / vel.w
    const real ri = (F == kF64) ? (real)pi.w : (real)wi.w;
    const real mi = (real)vi.w;
    const real kn = (real)kc.kn, kt = (real)kc.kt, mu = (real)kc.mu, two_zeta = (real)kc.two_zeta,
               neg_inv_kt = (real)kc.neg_inv_kt, dt = (real)kc.dt;
    const float cs_u = (float)g.cs;
    const uint32_t had = live ? hist.cnt_in[me] : 0u;
    const uint32_t ocnt = had & 0xFFu;
    for (uint32_t c = sub; c < ocnt; c += 4u) s_hid[p][c] = hist.id_in[(size_t)c * n + me];
    // the nine rows' candidate ranges, read at once
    uint32_t j0[9], len[9];
#pragma unroll
    for (int r = 0; r < 9; ++r) {
      const int zz = cr.cz + r / 3 - 1, yy = cr.cy + r % 3 - 1;
      const bool ok = live && zz >= 0 && zz < g.dims[2] && yy >= 0 && yy < g.dims[1];
      const uint32_t row = ok ? ((uint32_t)zz * (uint32_t)g.dims[1] + (uint32_t)yy) * (uint32_t)g.dims[0] : 0u;
      j0[r] = lb[row + (uint32_t)cr.x0];
      len[r] = ok ? lb[row + (uint32_t)cr.x1 + 1u] - j0[r] : 0u;
    }
    auto pair = [&](const G4& pj, real& dx, real& dy, real& dz) {
      if constexpr (F == kMixed) {
        probe_pair(pi, pj, cs_u, dx, dy, dz);
      } else {
        dx = pi.x - pj.x; dy = pi.y - pj.y; dz = pi.z - pj.z;
      }
    };
    // |d|^2: the FP64 unit rounds every operation; the mixed form's fused order is written out
    auto norm2 = [](real dx, real dy, real dz) {
      if constexpr (F == kMixed) return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
      else return dx * dx + dy * dy + dz * dz;
    };
    uint32_t nc = 0;
    auto test = [&](uint32_t j, bool cand, const G4& pj, const G4& wj) {
      real dx, dy, dz;
      pair(pj, dx, dy, dz);
      const real r2 = norm2(dx, dy, dz);
      const real rj = (F == kF64) ? (real)pj.w : (real)wj.w;
      const real R = ri + rj;
      const bool hit = cand && j != i && r2 < R * R && r2 > real(0.0);
      const uint32_t nib = (uint32_t)(__ballot(hit) >> qshift) & 15u;
      const uint32_t at = nc + (uint32_t)__popc(nib & below);
      if (hit && at < kDemList) s_list[p][at] = j;
      nc += (uint32_t)__popc(nib);
    };
    // rows three at a time, so that their first loads overlap
#pragma unroll
    for (int r0 = 0; r0 < 9; r0 += 3) {
      G4 pj[3], wj[3];
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const uint32_t j = sub < len[r0 + t] ? j0[r0 + t] + sub : self;
        pj[t] = gpos[j];
        if constexpr (F == kMixed) wj[t] = gom[j];
        else wj[t] = pj[t];   // unused: the FP64 radius is pos.w
      }
#pragma unroll
      for (int t = 0; t < 3; ++t) {
        const int r = r0 + t;
        test(j0[r] + sub, sub < len[r], pj[t], wj[t]);
        for (uint32_t b = sub + 4u; __ballot(b < len[r]) != 0ull; b += 4u) {
          const uint32_t j = b < len[r] ? j0[r] + b : self;
          const G4 q = gpos[j];
          G4 w = q;
          if constexpr (F == kMixed) w = gom[j];
          test(j, b < len[r], q, w);
        }
      }
    }
    real Fx = 0, Fy = 0, Fz = 0, Tx = 0, Ty = 0, Tz = 0;
    uint32_t walls = 0, nslip = 0;
    __builtin_amdgcn_wave_barrier();   // one wavefront: its LDS operations complete in order
    const uint32_t listed = nc < kDemList ? nc : kDemList;
    for (uint32_t t = sub; __ballot((t & ~3u) < listed) != 0ull; t += 4u) {
      real fx = 0, fy = 0, fz = 0, tx = 0, ty = 0, tz = 0;
      if (t < listed) {
        const uint32_t j = s_list[p][t];
        const G4 pj = gpos[j], vj = gvel[j], wj = gom[j];
        const uint32_t pid = ids[j];
        real dx, dy, dz;
        pair(pj, dx, dy, dz);
        real r2 = norm2(dx, dy, dz);
        const real rj = (F == kF64) ? (real)pj.w : (real)wj.w;
        real R = ri + rj;
        real d = sqrt(r2);
        real invd = real(1.0) / d;
        real nx = dx * invd, ny = dy * invd, nz = dz * invd;
        real delta = R - d;
        real wsx = ri * wi.x + rj * wj.x;
        real wsy = ri * wi.y + rj * wj.y;
        real wsz = ri * wi.z + rj * wj.z;
        real cx = wsy * nz - wsz * ny, cy = wsz * nx - wsx * nz, cz = wsx * ny - wsy * nx;
        real vrx = (vi.x - vj.x) - cx, vry = (vi.y - vj.y) - cy, vrz = (vi.z - vj.z) - cz;
        real vn = vrx * nx + vry * ny + vrz * nz;
        real vtx = vrx - vn * nx, vty = vry - vn * ny, vtz = vrz - vn * nz;
        real mj = (real)vj.w;
        real meff = mi * mj / (mi + mj);
        real cn = two_zeta * sqrt(meff * kn);
        real fn = kn * delta - cn * vn;
        uint32_t at = ocnt;
        for (uint32_t c = ocnt; c-- > 0u;) at = s_hid[p][c] == pid ? c : at;   // the first match
        real xox = 0, xoy = 0, xoz = 0;
        if (at < ocnt) {
          xox = xi_in[(size_t)(at * 3 + 0) * n + me];
          xoy = xi_in[(size_t)(at * 3 + 1) * n + me];
          xoz = xi_in[(size_t)(at * 3 + 2) * n + me];
        }
        real ft[3], xn[3];
        nslip += dem_tangential<real>(fn, nx, ny, nz, vtx, vty, vtz, xox, xoy, xoz, kt, mu, neg_inv_kt, dt, ft, xn);
        fx = fn * nx + ft[0];
        fy = fn * ny + ft[1];
        fz = fn * nz + ft[2];
        tx = ny * ft[2] - nz * ft[1], ty = nz * ft[0] - nx * ft[2], tz = nx * ft[1] - ny * ft[0];
        if (t < mc) {
          hist.id_out[(size_t)t * n + me] = pid;
          xi_out[(size_t)(t * 3 + 0) * n + me] = xn[0];
          xi_out[(size_t)(t * 3 + 1) * n + me] = xn[1];
          xi_out[(size_t)(t * 3 + 2) * n + me] = xn[2];
        }
      }
      for_quad([&](auto K) {
        const real ax = quad_bcast<K.value>(fx), ay = quad_bcast<K.value>(fy), az = quad_bcast<K.value>(fz);
        const real bx = quad_bcast<K.value>(tx), by = quad_bcast<K.value>(ty), bz = quad_bcast<K.value>(tz);
        if ((t & ~3u) + (uint32_t)K.value < listed) {
          Fx = Fx + ax;
          Fy = Fy + ay;
          Fz = Fz + az;
          Tx = Tx - ri * bx; Ty = Ty - ri * by; Tz = Tz - ri * bz;
        }
      });
    }
    nslip += quad_bcast<1>(nslip) + quad_bcast<2>(nslip) + quad_bcast<3>(nslip);   // lane 0's sum is used
    if (live) {
      const double4 xs = spos[i], vs = svel[i], ws = som[i];   // (not held through the contacts)
      // walls: bit 2a = lower wall of axis a (normal +e_a), bit 2a+1 = upper
      // (-e_a); the quad's lanes compute the same, each stores its share
      for (int w = 0; w < 6; ++w) {
        const bool store = (uint32_t)(w & 3) == sub;
        real delta = real(-1.0);
        if (kc.wall_mask & (1u << w)) {
          int a = w >> 1;
          double pa = a == 0 ? xs.x : (a == 1 ? xs.y : xs.z);
          double dist = (w & 1) ? (kc.wall_hi[a] - pa) : (pa - kc.wall_lo[a]);
          if constexpr (F == kF64) delta = ri - dist;
          else delta = (real)(xs.w - dist);
        }
        if (!(delta > real(0.0))) continue;
        int a = w >> 1;
        real sg = (w & 1) ? real(-1.0) : real(1.0);
        real nx = a == 0 ? sg : real(0.0), ny = a == 1 ? sg : real(0.0), nz = a == 2 ? sg : real(0.0);
        real wsx = ri * wi.x, wsy = ri * wi.y, wsz = ri * wi.z;
        real cx = wsy * nz - wsz * ny, cy = wsz * nx - wsx * nz, cz = wsx * ny - wsy * nx;
        real vrx = vi.x - cx, vry = vi.y - cy, vrz = vi.z - cz;
        real vn = vrx * nx + vry * ny + vrz * nz;
        real vtx = vrx - vn * nx, vty = vry - vn * ny, vtz = vrz - vn * nz;
        real cn = two_zeta * sqrt(mi * kn);
        real fn = kn * delta - cn * vn;
        real xox = 0, xoy = 0, xoz = 0;
        if ((had >> (8 + w)) & 1u) {
          xox = wxi_in[(size_t)(w * 3 + 0) * n + me];
          xoy = wxi_in[(size_t)(w * 3 + 1) * n + me];
          xoz = wxi_in[(size_t)(w * 3 + 2) * n + me];
        }
        real ft[3], xn[3];
        nslip += dem_tangential<real>(fn, nx, ny, nz, vtx, vty, vtz, xox, xoy, xoz, kt, mu, neg_inv_kt, dt, ft, xn);
        walls |= 1u << w;
        Fx = Fx + (fn * nx + ft[0]);
        Fy = Fy + (fn * ny + ft[1]);
        Fz = Fz + (fn * nz + ft[2]);
        real tx = ny * ft[2] - nz * ft[1], ty = nz * ft[0] - nx * ft[2], tz = nx * ft[1] - ny * ft[0];
        Tx = Tx - ri * tx; Ty = Ty - ri * ty; Tz = Tz - ri * tz;
        if (store) {
          wxi_out[(size_t)(w * 3 + 0) * n + me] = xn[0];
          wxi_out[(size_t)(w * 3 + 1) * n + me] = xn[1];
          wxi_out[(size_t)(w * 3 + 2) * n + me] = xn[2];
        }
      }
      // symplectic Euler in FP64
      const double m64 = vs.w, r64 = xs.w;
      double axx = (double)Fx / m64 + kc.g[0];
      double ayy = (double)Fy / m64 + kc.g[1];
      double azz = (double)Fz / m64 + kc.g[2];
      double4 v2 = vs, x2 = xs, w2 = ws;
      v2.x = vs.x + kc.dt * axx;
      v2.y = vs.y + kc.dt * ayy;
      v2.z = vs.z + kc.dt * azz;
      x2.x = xs.x + kc.dt * v2.x;
      x2.y = xs.y + kc.dt * v2.y;
      x2.z = xs.z + kc.dt * v2.z;
      double inertia = 0.4 * m64 * r64 * r64;
      w2.x = ws.x + kc.dt * ((double)Tx / inertia);
      w2.y = ws.y + kc.dt * ((double)Ty / inertia);
      w2.z = ws.z + kc.dt * ((double)Tz / inertia);
      double fx = floor((x2.x - g.lo[0]) * g.inv_cs);
      double fy = floor((x2.y - g.lo[1]) * g.inv_cs);
      double fz = floor((x2.z - g.lo[2]) * g.inv_cs);
      const bool ok = fx >= 0.0 && fy >= 0.0 && fz >= 0.0 && fx < (double)g.dims[0] &&
                      fy < (double)g.dims[1] && fz < (double)g.dims[2];
      if (sub == 0u) {
        uint32_t key = key_i;   // a sphere outside the grid keeps its cell
        if (ok) key = ((uint32_t)fz * (uint32_t)g.dims[1] + (uint32_t)fy) * (uint32_t)g.dims[0] + (uint32_t)fx;
        const bool runaway = (v2.x * v2.x + v2.y * v2.y + v2.z * v2.z) * (kc.dt * kc.dt) > 0.0625 * (r64 * r64);
        mv = move_to_cell(moved, i, key_i, key, runaway);
        opos[i] = x2;
        ovel[i] = v2;
        oom[i] = w2;
        if (oforce) oforce[i] = make_double4(axx, ayy, azz, 0.0);
        okeys[i] = key;
        hist.cnt_out[me] = (nc < mc ? nc : mc) | walls << 8;
        if (nc > mc) atomicOr(&flags[FLAG_CAPACITY], 1u);
        if (events) {   // step-weighted fingerprints of this particle's contact and slip events
          events[me] += ev_weight * (nc + (uint32_t)__popc(walls));
          events[(size_t)n + me] += ev_weight * nslip;
        }
        if (!isfinite(axx) || !isfinite(ayy) || !isfinite(azz)) atomicOr(&flags[FLAG_NONFINITE], 1u);
        if (runaway) atomicOr(&flags[FLAG_CFL], 1u);
        if (!ok) atomicOr(&flags[FLAG_DOMAIN], 1u);
      }
    }
  }
  moved_word_quad(moved, tile, mv);
}

template <int F>
void dem_step_impl(Ctx& c) {
  using G4 = typename DemForm<F>::G4;
  using real = typename DemForm<F>::real;
  neighbors_build(c);
  const uint32_t n = (uint32_t)c.n;
  if (!n) return;
  const G4* gpos = (F == kMixed) ? c.off32.as<G4>() : c.pos[c.cur].as<G4>();
  const G4* gvel = (F == kMixed) ? c.vel32.as<G4>() : c.vel[c.cur].as<G4>();
  const G4* gom = (F == kMixed) ? c.om32.as<G4>() : c.omega[c.cur].as<G4>();
  const int h = c.cur_hist;
  DemHist hist{c.hcnt[h].as<uint32_t>(), c.hid[h].as<uint32_t>(), c.hxi[h].p, c.wxi[h].p,
               c.hcnt[h ^ 1].as<uint32_t>(), c.hid[h ^ 1].as<uint32_t>(), c.hxi[h ^ 1].p, c.wxi[h ^ 1].p};
  const uint32_t n_tiles = blocks_for(n, (int)kQuadSlots);
  const double ge = (double)sizeof(real);
  const double lb_bytes = 4.0 * (double)c.grid.n_cells / (double)n;
  // gathered: pos 3 + r, vel 3 + m, omega 3; ids + key; state in/out (pos, vel, omega) 3 x 24 x 2;
  // history in/out: count + (typical) 6 slots x (id + 3 reals); wall springs move for
  // the few spheres that touch a wall only
  double hist_bytes = 2.0 * (4.0 + 6.0 * (4.0 + 3.0 * ge));
  double bytes = (11.0 * ge + 8.0 + lb_bytes + 2.0 * 3.0 * 32.0 + 4.0 + hist_bytes) * n;
  LaunchScope ls(&c, F == kF64 ? "dem_force_f64" : "dem_force_mixed", bytes);
  const int dst = c.cur ^ 1, kdst = c.cur_key ^ 1;
  k_dem_force<F><<<tile_grid(n_tiles), 64, 0, c.stream>>>(
      n, c.n_moving, gpos, gvel, gom, c.ids[c.cur_ids].as<uint32_t>(), c.keys[c.cur_key].as<uint32_t>(),
      c.lb.as<uint32_t>(), c.grid, c.dem, c.pos[c.cur].as<double4>(), c.vel[c.cur].as<double4>(),
      c.omega[c.cur].as<double4>(), c.pos[dst].as<double4>(), c.vel[dst].as<double4>(),
      c.omega[dst].as<double4>(), c.keys[kdst].as<uint32_t>(), c.keep_acc ? c.acc.as<double4>() : nullptr,
      hist, moved_out(c), c.flags.as<uint32_t>(),
      c.ev_weight ? c.events.as<uint32_t>() : nullptr, c.ev_weight, n_tiles);
  PR_HIP(hipGetLastError());
  c.cur = dst;
  c.cur_key = kdst;
  c.cur_hist ^= 1;
  c.sorted = false;
  c.keys_valid = true;
  c.inc_ready = true;   // keys[cur_key ^ 1] and lb still describe the slots the step kept
}

}  // namespace prestige
