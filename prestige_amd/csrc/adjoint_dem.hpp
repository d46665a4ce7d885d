// adjoint_dem.hpp — reverse mode of one DEM step, gather form.
//
// Forward row (i, j) of a contact, evaluated by particle i (dem_kernels.hpp):
//   d = x_i - x_j, r = |d|, n = d/r, delta = R - r,
//   ws = r_i w_i + r_j w_j, vr = (v_i - v_j) - ws x n, vn = vr.n,
//   vt = vr - vn n, cn = tz sqrt(meff kn), fn = kn delta - cn vn,
//   xp = xo - (xo.n) n, x0 = xp + dt vt, ft0 = -kt x0,
//   slip (|ft0| > mu |fn|): ft = ft0 mu|fn|/|ft0|, xn = -ft/kt;  else ft = ft0, xn = x0,
//   F_i += fn n + ft,  T_i += -r_i (n x ft),  history xn stored at i for j.
// Walls: the same row with the partner terms removed, n = +-e_a and
// delta = r_i - dist, m_eff = m_i.  Integrator: a = F/m + g, v' = v + dt a,
// x' = x + dt v', w' = w + dt T/I.
//
// Reverse: each particle k walks its own frozen contact list of the step
// (the history it wrote, in forward order; ids -> slots through the inverse
// permutation) and, for every partner j, runs the vector-Jacobian product of
// its own row (k, j) with seeds (Fbar_k, Tbar_k, xibar of its history copy)
// and of the partner's row (j, k) with the partner's seeds, keeping only the
// terms that belong to k.  Both history copies of a contact therefore get
// their own adjoint from their owner, the parameter sums take own rows only,
// and nothing is scattered: no atomics.  kt = (kt0/kn0) kn moves with kn;
// tz = 2 zeta(e) with dtz/de from the host.  Arithmetic is FP64 on the FP64
// state for both forms; the contact set and the history slots are the
// forward's own.
#pragma once
#include "dem_kernels.hpp"

namespace prestige {

struct DemAdjConst {
  double kn, kt, mu, tz, dtz_de, dt, kt_per_kn;
  double wall_lo[3], wall_hi[3];
  uint32_t wall_mask, max_contacts;
};

struct V3 {
  double x, y, z;
};
__device__ inline V3 v3(double x, double y, double z) { return V3{x, y, z}; }
__device__ inline V3 operator+(V3 a, V3 b) { return v3(a.x + b.x, a.y + b.y, a.z + b.z); }
__device__ inline V3 operator-(V3 a, V3 b) { return v3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ inline V3 operator*(double s, V3 a) { return v3(s * a.x, s * a.y, s * a.z); }
__device__ inline double dot(V3 a, V3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ inline V3 cross(V3 a, V3 b) {
  return v3(a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x);
}
__device__ inline V3 xyz(const double4& a) { return v3(a.x, a.y, a.z); }

// Gradients of one contact row.
struct RowBar {
  V3 d;                  // w.r.t. the pair vector d (pairs) / position of i (walls)
  V3 vi, vj, wi, wj;     // w.r.t. velocities and angular velocities
  V3 xo;                 // w.r.t. the incoming tangential spring
  double kn, tz, mu;     // w.r.t. parameters (kt folded into kn)
};

// VJP of one row.  wall = true: n is the wall normal (no dependence on d),
// delta = ri - dist, and the partner terms vanish.
__device__ inline RowBar row_vjp(bool wall, V3 d, V3 nwall, double delta_wall, V3 vi, V3 vj, V3 wi, V3 wj,
                                 double ri, double rj, double mi, double mj, V3 xo, V3 Fb, V3 Tb, V3 xnb,
                                 const DemAdjConst& k) {
  // ---- forward recompute ----
  V3 n;
  double r = 0.0, invr = 0.0, delta;
  if (wall) {
    n = nwall;
    delta = delta_wall;
  } else {
    r = sqrt(dot(d, d));
    invr = 1.0 / r;
    n = invr * d;
    delta = (ri + rj) - r;
  }
  const V3 ws = wall ? ri * wi : ri * wi + rj * wj;
  const V3 cr = cross(ws, n);
  const V3 vr = (wall ? vi : vi - vj) - cr;
  const double vn = dot(vr, n);
  const V3 vt = vr - vn * n;
  const double meff = wall ? mi : mi * mj / (mi + mj);
  const double sq = sqrt(meff * k.kn);
  const double cn = k.tz * sq;
  const double fn = k.kn * delta - cn * vn;
  const double s = dot(xo, n);
  const V3 xp = xo - s * n;
  const V3 x0 = xp + k.dt * vt;
  const V3 ft0 = (-k.kt) * x0;
  const double ftn = sqrt(dot(ft0, ft0));
  const double sg = fn < 0.0 ? -1.0 : 1.0;
  const double fcap = k.mu * sg * fn;
  const bool slip = ftn > fcap;
  const double sc = slip ? fcap / ftn : 1.0;
  const V3 ft = sc * ft0;
  // ---- reverse ----
  RowBar b{};
  V3 nb = v3(0, 0, 0), ftb = v3(0, 0, 0);
  // T = -ri (n x ft)
  const V3 tqb = (-ri) * Tb;
  nb = nb + cross(ft, tqb);
  ftb = ftb + cross(tqb, n);
  // F = fn n + ft
  double fnb = dot(Fb, n);
  nb = nb + fn * Fb;
  ftb = ftb + Fb;
  V3 ft0b, x0b;
  double ktb = 0.0;
  if (slip) {
    // xn = ft * (-1/kt)
    ftb = ftb + (-1.0 / k.kt) * xnb;
    ktb += dot(xnb, ft) / (k.kt * k.kt);
    ft0b = sc * ftb;
    const double scb = dot(ftb, ft0);
    const double fcapb = scb / ftn;
    const double ftnb = -scb * fcap / (ftn * ftn);
    ft0b = ft0b + (ftnb / ftn) * ft0;
    b.mu += fcapb * sg * fn;
    fnb += fcapb * k.mu * sg;
    x0b = v3(0, 0, 0);
  } else {
    ft0b = ftb;
    x0b = xnb;
  }
  // ft0 = -kt x0
  x0b = x0b + (-k.kt) * ft0b;
  ktb += -dot(ft0b, x0);
  // x0 = xp + dt vt
  const V3 xpb = x0b;
  V3 vtb = k.dt * x0b;
  // xp = xo - s n, s = xo.n
  b.xo = xpb;
  const double sb = -dot(xpb, n);
  nb = nb + (-s) * xpb;
  b.xo = b.xo + sb * n;
  nb = nb + sb * xo;
  // fn = kn delta - cn vn
  b.kn += fnb * delta;
  const double deltab = fnb * k.kn;
  const double cnb = -fnb * vn;
  double vnb = -fnb * cn;
  // cn = tz sqrt(meff kn)
  b.tz += cnb * sq;
  if (k.kn > 0.0) b.kn += cnb * cn / (2.0 * k.kn);
  // vt = vr - vn n
  V3 vrb = vtb;
  vnb += -dot(vtb, n);
  nb = nb + (-vn) * vtb;
  // vn = vr . n
  vrb = vrb + vnb * n;
  nb = nb + vnb * vr;
  // vr = (vi - vj) - cr
  b.vi = vrb;
  b.vj = (-1.0) * vrb;
  const V3 crb = (-1.0) * vrb;
  // cr = ws x n
  const V3 wsb = cross(n, crb);
  nb = nb + cross(crb, ws);
  b.wi = ri * wsb;
  b.wj = rj * wsb;
  // geometry
  if (wall) {
    // delta = ri - dist with d(dist)/dx_i = n: ddelta/dx_i = -n
    b.d = (-deltab) * n;
    b.vj = v3(0, 0, 0);
    b.wj = v3(0, 0, 0);
  } else {
    // n = d / r, delta = R - r
    const V3 dn = invr * (nb - dot(nb, n) * n);
    b.d = dn + (-deltab) * n;
  }
  b.kn += ktb * k.kt_per_kn;
  return b;
}

// Index of partner among the owner's cnt contacts (-1: none), eight ids read
// at a time.
__device__ inline int find_slot(const uint32_t* __restrict__ hid, uint32_t cnt, uint32_t n, uint32_t owner,
                                uint32_t partner) {
  for (uint32_t c0 = 0; c0 < cnt; c0 += 8u) {
    uint32_t id[8];
#pragma unroll
    for (uint32_t u = 0; u < 8u; ++u) id[u] = hid[(size_t)(c0 + u < cnt ? c0 + u : c0) * n + owner];
    int at = -1;
#pragma unroll
    for (uint32_t u = 8u; u-- > 0u;)
      if (c0 + u < cnt && id[u] == partner) at = (int)(c0 + u);
    if (at >= 0) return at;
  }
  return -1;
}

template <class H>
__device__ inline V3 load_xi(const H* __restrict__ xi, uint32_t slot, uint32_t n, uint32_t owner) {
  return v3((double)xi[(size_t)(slot * 3 + 0) * n + owner], (double)xi[(size_t)(slot * 3 + 1) * n + owner],
            (double)xi[(size_t)(slot * 3 + 2) * n + owner]);
}

__device__ inline void store3(double* __restrict__ a, uint32_t slot, uint32_t n, uint32_t owner, V3 v) {
  a[(size_t)(slot * 3 + 0) * n + owner] = v.x;
  a[(size_t)(slot * 3 + 1) * n + owner] = v.y;
  a[(size_t)(slot * 3 + 2) * n + owner] = v.z;
}

__device__ inline V3 load3(const double* __restrict__ a, uint32_t slot, uint32_t n, uint32_t owner) {
  return v3(a[(size_t)(slot * 3 + 0) * n + owner], a[(size_t)(slot * 3 + 1) * n + owner],
            a[(size_t)(slot * 3 + 2) * n + owner]);
}

struct DemStepView {
  const double4 *pos, *vel, *om;       // FP64 sorted pre-step state (pos.w radius, vel.w mass)
  const uint32_t *ids, *perm, *slot_of;
  const uint32_t *cnt_in, *hid_in;     // history the step read
  const void* xi_in;
  const void* wxi_in;
  const uint32_t *cnt_out, *hid_out;   // contacts the step found (its frozen list)
};

// vbt = vbar' + dt xbar', Fbar = dt vbt / m, Tbar = dt wbar' / I; and the slot of
// each id.
static __global__ __launch_bounds__(kBlock) void k_dem_adj_prep(uint32_t n, uint64_t n_moving, DemStepView s,
                                                                 const double4* __restrict__ xb,
                                                                 double4* __restrict__ vb,
                                                                 const double4* __restrict__ wb,
                                                                 double4* __restrict__ Fb, double4* __restrict__ Tb,
                                                                 double dt, uint32_t* __restrict__ slot_of) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const uint32_t id = s.ids[k];
  slot_of[id] = k;
  if ((uint64_t)id >= n_moving) {
    vb[k] = make_double4(0, 0, 0, 0);
    Fb[k] = make_double4(0, 0, 0, 0);
    Tb[k] = make_double4(0, 0, 0, 0);
    return;
  }
  const double m = s.vel[k].w, r = s.pos[k].w;
  const double4 x = xb[k], v = vb[k], w = wb[k];
  const double4 vt = make_double4(v.x + dt * x.x, v.y + dt * x.y, v.z + dt * x.z, 0.0);
  vb[k] = vt;
  const double fm = dt / m;
  Fb[k] = make_double4(fm * vt.x, fm * vt.y, fm * vt.z, 0.0);
  const double ti = dt / (0.4 * m * r * r);
  Tb[k] = make_double4(ti * w.x, ti * w.y, ti * w.z, 0.0);
}

// Contact adjoint + integrator assembly for one reverse step, four lanes per
// particle (a quad): each lane takes one of the particle's contacts at a time,
// the quad's sums are added in lane order.  A contact is two row products of
// some 200 FP64 operations behind a chain of reads (partner id, its slot, its
// state, three searches); with one lane per particle 20,000 spheres were 313
// wavefronts that ran their contacts in turn: 40 us, 18 with quads.
template <class H>
__global__ __launch_bounds__(64) void k_dem_adj(uint32_t n, uint64_t n_moving, DemStepView s, DemAdjConst kc,
                                                const double4* __restrict__ xb_in,
                                                const double4* __restrict__ vb_in,
                                                const double4* __restrict__ wb_in,
                                                const double4* __restrict__ Fb, const double4* __restrict__ Tb,
                                                const double* __restrict__ hb_next,
                                                const double* __restrict__ wallb_next,
                                                const uint32_t* __restrict__ wallm_next,
                                                double* __restrict__ hb_prev, double* __restrict__ wallb_prev,
                                                uint32_t* __restrict__ wallm_prev,
                                                double4* __restrict__ xb_out, double4* __restrict__ vb_out,
                                                double4* __restrict__ wb_out, double4* __restrict__ partial,
                                                uint32_t n_tiles) {
  __shared__ uint32_t s_had[kQuadSlots];   // history slots a contact of the step continues
  const uint32_t tile = xcd_tile(blockIdx.x);
  if (tile >= n_tiles) return;
  const H* xi_in = (const H*)s.xi_in;
  const H* wxi_in = (const H*)s.wxi_in;
  const uint32_t lane = threadIdx.x, sub = lane & 3u, p = lane >> 2;
  const uint32_t k = tile * kQuadSlots + p;
  const bool in = k < n;
  const uint32_t self = in ? k : tile * kQuadSlots;
  const uint32_t me = s.ids[self], dst = s.perm[self];
  const bool live = in && (uint64_t)me < n_moving;
  const uint32_t had_in = in ? s.cnt_in[me] : 0u;   // contacts and walls (DemHist)
  const uint32_t cin = had_in & 0xFFu, cout = live ? s.cnt_out[me] & 0xFFu : 0u;
  double pk = 0.0, pt = 0.0, pm = 0.0;
  V3 X = v3(0, 0, 0), V = v3(0, 0, 0), W = v3(0, 0, 0);
  if (sub == 0u) s_had[p] = 0u;
  wave_lds_fence();
  const double4 pk4 = s.pos[self], vk4 = s.vel[self], wk4 = s.om[self];
  const V3 xk = xyz(pk4), vk = xyz(vk4), wk = xyz(wk4);
  const double rk = pk4.w, mk = vk4.w;
  const V3 Fbk = xyz(Fb[self]), Tbk = xyz(Tb[self]);
  for (uint32_t c = sub; c < cout; c += 4u) {
    const uint32_t pid = s.hid_out[(size_t)c * n + me];
    const uint32_t j = s.slot_of[pid];
    const uint32_t cjin = s.cnt_in[pid] & 0xFFu, cjout = s.cnt_out[pid] & 0xFFu;
    const double4 pj4 = s.pos[j], vj4 = s.vel[j], wj4 = s.om[j];
    const bool jm = (uint64_t)pid < n_moving;
    const V3 Fbj = jm ? xyz(Fb[j]) : v3(0, 0, 0), Tbj = jm ? xyz(Tb[j]) : v3(0, 0, 0);
    const V3 xj = xyz(pj4), vj = xyz(vj4), wj = xyz(wj4);
    const double rj = pj4.w, mj = vj4.w;
    const int ci = find_slot(s.hid_in, cin, n, me, pid);
    const int cj = find_slot(s.hid_in, cjin, n, pid, me);
    const int co = find_slot(s.hid_out, cjout, n, pid, me);
    // own row (k, j)
    const V3 xo = ci >= 0 ? load_xi(xi_in, (uint32_t)ci, n, me) : v3(0, 0, 0);
    const V3 xnb = load3(hb_next, c, n, me);
    const RowBar a = row_vjp(false, xk - xj, v3(0, 0, 0), 0.0, vk, vj, wk, wj, rk, rj, mk, mj, xo, Fbk, Tbk, xnb, kc);
    X = X + a.d;
    V = V + a.vi;
    W = W + a.wi;
    if (ci >= 0) {
      store3(hb_prev, (uint32_t)ci, n, me, a.xo);
      atomicOr(&s_had[p], 1u << ci);   // max_contacts <= 32
    }
    pk += a.kn;
    pt += a.tz;
    pm += a.mu;
    // partner row (j, k): keep the terms of k
    const V3 xoj = cj >= 0 ? load_xi(xi_in, (uint32_t)cj, n, pid) : v3(0, 0, 0);
    const V3 xnbj = co >= 0 ? load3(hb_next, (uint32_t)co, n, pid) : v3(0, 0, 0);
    const RowBar b = row_vjp(false, xj - xk, v3(0, 0, 0), 0.0, vj, vk, wj, wk, rj, rk, mj, mk, xoj, Fbj, Tbj, xnbj, kc);
    X = X - b.d;
    V = V + b.vj;
    W = W + b.wj;
  }
  wave_lds_fence();
  // history slots no contact continues get zero adjoints
  const uint32_t had = s_had[p];
  for (uint32_t c = sub; c < cin; c += 4u)
    if (!((had >> c) & 1u)) store3(hb_prev, c, n, me, v3(0, 0, 0));
  // the quad's sums, in lane order, in all its lanes
  auto quad_sum = [](double v) {
    return ((quad_bcast<0>(v) + quad_bcast<1>(v)) + quad_bcast<2>(v)) + quad_bcast<3>(v);
  };
  auto quad_sum3 = [&](V3 v) { return v3(quad_sum(v.x), quad_sum(v.y), quad_sum(v.z)); };
  X = quad_sum3(X);
  V = quad_sum3(V);
  W = quad_sum3(W);
  if (in) {
    // walls: the quad's lanes compute the same, each stores its share.  The
    // spring of a wall has an adjoint where the step touched the wall (wallm);
    // every other is zero and neither written nor read (100,000 mixed spheres
    // with few contacts: 26 -> 23 us a pass).
    const uint32_t later = wallm_next[me];
    uint32_t walls = 0;
    for (int w = 0; w < 6; ++w) {
      bool on = false;
      double delta = 0.0;
      V3 nw = v3(0, 0, 0);
      if (live && (kc.wall_mask & (1u << w))) {
        const int ax = w >> 1;
        const double pa = ax == 0 ? xk.x : (ax == 1 ? xk.y : xk.z);
        const double dist = (w & 1) ? (kc.wall_hi[ax] - pa) : (pa - kc.wall_lo[ax]);
        delta = rk - dist;
        on = delta > 0.0;
        const double sgn = (w & 1) ? -1.0 : 1.0;
        nw = v3(ax == 0 ? sgn : 0.0, ax == 1 ? sgn : 0.0, ax == 2 ? sgn : 0.0);
      }
      if (on) {
        const V3 xo = (had_in >> (8 + w)) & 1u ? load_xi(wxi_in, (uint32_t)w, n, me) : v3(0, 0, 0);
        const V3 xnb = (later >> w) & 1u ? load3(wallb_next, (uint32_t)w, n, me) : v3(0, 0, 0);
        const RowBar a = row_vjp(true, v3(0, 0, 0), nw, delta, vk, v3(0, 0, 0), wk, v3(0, 0, 0), rk, 0.0, mk, 0.0, xo,
                                 Fbk, Tbk, xnb, kc);
        X = X + a.d;
        V = V + a.vi;
        W = W + a.wi;
        walls |= 1u << w;
        if ((uint32_t)(w & 3) == sub) store3(wallb_prev, (uint32_t)w, n, me, a.xo);
        if (sub == 0u) {
          pk += a.kn;
          pt += a.tz;
          pm += a.mu;
        }
      }
    }
    if (sub == 0u) wallm_prev[me] = walls;
    const V3 z = v3(0, 0, 0);
    if (sub < 3u) {
      const double4* from = sub == 0u ? xb_in : (sub == 1u ? vb_in : wb_in);
      double4* to = sub == 0u ? xb_out : (sub == 1u ? vb_out : wb_out);
      const V3 d = sub == 0u ? X : (sub == 1u ? V : W);
      const double4 v0 = from[k];
      const V3 r = live ? v3(v0.x + d.x, v0.y + d.y, v0.z + d.z) : z;
      to[dst] = make_double4(r.x, r.y, r.z, 0.0);
    }
  }
  pt *= kc.dtz_de;
  for (int o = 32; o > 0; o >>= 1) {
    pk += __shfl_down(pk, (unsigned)o, 64);
    pt += __shfl_down(pt, (unsigned)o, 64);
    pm += __shfl_down(pm, (unsigned)o, 64);
  }
  if (lane == 0u) partial[tile] = make_double4(pk, pt, pm, 0.0);
}

// Parameter sums of one reverse step per block (its partials lie nparts apart
// per step), in a fixed order, into its first partial.
static __global__ void k_dem_adj_reduce(uint32_t nparts, double4* __restrict__ partial) {
  __shared__ double s[3][256];
  double4* part = partial + (size_t)blockIdx.x * nparts;
  double a = 0.0, b = 0.0, c = 0.0;
  for (uint32_t q = threadIdx.x; q < nparts; q += blockDim.x) {
    const double4 v = part[q];
    a += v.x;
    b += v.y;
    c += v.z;
  }
  s[0][threadIdx.x] = a;
  s[1][threadIdx.x] = b;
  s[2][threadIdx.x] = c;
  __syncthreads();
  for (uint32_t st = blockDim.x / 2; st > 0; st >>= 1) {
    if (threadIdx.x < st)
      for (int k = 0; k < 3; ++k) s[k][threadIdx.x] += s[k][threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[0] = make_double4(s[0][0], s[1][0], s[2][0], 0.0);
}

// acc[0..2] += the sums of `steps` reverse steps, step by step.
static __global__ void k_dem_adj_acc(uint32_t nparts, uint32_t steps, const double4* __restrict__ partial,
                                     double* __restrict__ acc) {
  double a = acc[0], b = acc[1], c = acc[2];
  for (uint32_t t = 0; t < steps; ++t) {
    const double4 v = partial[(size_t)t * nparts];
    a += v.x;
    b += v.y;
    c += v.z;
  }
  acc[0] = a;
  acc[1] = b;
  acc[2] = c;
}

}  // namespace prestige

namespace prestige {

void snapshot_state(Ctx& c, Snapshot& s);
void restore_state(Ctx& c, Snapshot& s);
void copy_many(Ctx& c, const std::vector<Copy>& list);
void adj_seed_gather(Ctx& c, const uint32_t* ids, const double* seed_x, const double* seed_v);
void adj_grad_scatter(Ctx& c, const uint32_t* ids, const double4* vb, double* grad_v0_host);
void ensure_adj_buffers(Ctx& c);

// Keep what the reverse sweep needs from step t of a segment, which just ran,
// in rec[t].  Taken by swap (the next step overwrites them before reading): the
// sorted pre-step state, the permutation, the contact history the step read and
// the previous step's ids, whose order this step's build left.  The history a
// step writes is the one the next step reads, so rec[t + 1] holds step t's
// contacts; the segment's last step copies both.
template <class H>
void record_dem_step(Ctx& c, Tape& T, uint32_t t, bool last) {
  StepRecord& r = *T.rec[t];
  const size_t n = c.n ? c.n : 1, mc = c.desc.max_contacts;
  const int prev = c.cur ^ 1, hin = c.cur_hist ^ 1, hout = c.cur_hist;
  take_buffer(c.pos[prev], r.state_pos);
  take_buffer(c.vel[prev], r.state_vel);
  take_buffer(c.omega[prev], r.state_om);
  take_buffer(c.vals[c.perm_buf], r.perm);
  take_buffer(c.hcnt[hin], r.hcnt);
  take_buffer(c.hid[hin], r.hid);
  take_buffer(c.hxi[hin], r.hxi);
  take_buffer(c.wxi[hin], r.wxi);
  if (t > 0) take_buffer(c.ids[c.cur_ids ^ 1], T.rec[t - 1]->ids);
  if (!last) return;
  copy_many(c, {{&r.ids, &c.ids[c.cur_ids], n * 4}, {&r.hcnt_out, &c.hcnt[hout], n * 4},
                {&r.hid_out, &c.hid[hout], n * mc * 4}});
}

inline DemAdjConst dem_adj_const(const Ctx& c) {
  DemAdjConst k{};
  k.kn = c.dem.kn;
  k.kt = c.dem.kt;
  k.mu = c.dem.mu;
  k.tz = c.dem.two_zeta;
  const double L = std::log(c.desc.restitution);
  const double s = M_PI * M_PI + L * L;
  k.dtz_de = 2.0 * (-M_PI * M_PI / (s * std::sqrt(s) * c.desc.restitution));
  k.dt = c.dem.dt;
  k.kt_per_kn = c.dem.kn > 0.0 ? c.dem.kt / c.dem.kn : 0.0;
  for (int a = 0; a < 3; ++a) {
    k.wall_lo[a] = c.dem.wall_lo[a];
    k.wall_hi[a] = c.dem.wall_hi[a];
  }
  k.wall_mask = c.dem.wall_mask;
  k.max_contacts = c.dem.max_contacts;
  return k;
}

template <int F>
void dem_tape_forward(Ctx& c, uint32_t nsteps, uint32_t every) {
  using H = typename std::conditional<F == kF64, double, float>::type;
  Tape& T = c.tape;
  T.clear();
  T.nsteps = nsteps;
  T.every = every;
  // the last segment is recorded on the way, so the reverse sweep starts
  // without recomputing it
  const uint32_t last0 = nsteps ? ((nsteps - 1) / every) * every : 0;
  while (T.rec.size() < every) T.rec.emplace_back(new StepRecord());
  for (uint32_t s = 0; s < nsteps; ++s) {
    if (s % every == 0) {
      snapshot_state(c, T.next_ckpt());
    }
    dem_step_impl<F>(c);
    if (s >= last0) record_dem_step<H>(c, T, s - last0, s + 1 == nsteps);
  }
  T.last_recorded = nsteps > 0;
  if (!c.tape.final_state) c.tape.final_state.reset(new Snapshot());
  snapshot_state(c, *c.tape.final_state);
  c.check_flags();
  c.tape.valid = true;
}

template <int F, class H>
void dem_adjoint(Ctx& c, const double* seed_x, const double* seed_v, double* grad_params, double* grad_v0) {
  Tape& T = c.tape;
  const uint32_t n = (uint32_t)c.n;
  const size_t nn = n ? n : 1, mc = c.desc.max_contacts;
  const uint32_t nb = blocks_for(n), tiles = blocks_for(n, (int)kQuadSlots);
  ensure_adj_buffers(c);
  T.partial.alloc((size_t)tiles * std::min(T.every, T.nsteps) * sizeof(double4) + 64);
  T.hb[0].alloc(nn * mc * 3 * sizeof(double));
  T.hb[1].alloc(nn * mc * 3 * sizeof(double));
  T.wallb[0].alloc(nn * 18 * sizeof(double));
  T.wallb[1].alloc(nn * 18 * sizeof(double));
  for (DevBuf& b : T.wallm) b.alloc(nn * 4);
  T.slot_of.alloc(nn * 4);
  PR_HIP(hipMemsetAsync(T.acc.p, 0, 3 * sizeof(double), c.stream));
  PR_HIP(hipMemsetAsync(T.wb.p, 0, nn * sizeof(double4), c.stream));
  PR_HIP(hipMemsetAsync(T.hb[0].p, 0, nn * mc * 3 * sizeof(double), c.stream));
  PR_HIP(hipMemsetAsync(T.wallm[0].p, 0, nn * 4, c.stream));
  adj_seed_gather(c, T.final_state->ids.as<uint32_t>(), seed_x, seed_v);
  double4 *xb = T.xb.as<double4>(), *vb = T.vb.as<double4>(), *wb = T.wb.as<double4>();
  double4 *xb2 = T.xb2.as<double4>(), *vb2 = T.vb2.as<double4>(), *wb2 = T.wb2.as<double4>();
  double *hn = T.hb[0].as<double>(), *hp = T.hb[1].as<double>();
  double *wn = T.wallb[0].as<double>(), *wp = T.wallb[1].as<double>();
  uint32_t *mn = T.wallm[0].as<uint32_t>(), *mp = T.wallm[1].as<uint32_t>();
  const DemAdjConst kc = dem_adj_const(c);
  const uint32_t nseg = (T.nsteps + T.every - 1) / T.every;
  while (T.rec.size() < T.every) T.rec.emplace_back(new StepRecord());
  for (uint32_t seg = nseg; seg-- > 0;) {
    const uint32_t s0 = seg * T.every;
    const uint32_t len = (T.nsteps - s0) < T.every ? (T.nsteps - s0) : T.every;
    if (!(seg == nseg - 1 && T.last_recorded)) {
      restore_state(c, *T.ckpt[seg]);
      for (uint32_t t = 0; t < len; ++t) {
        dem_step_impl<F>(c);
        record_dem_step<H>(c, T, t, t + 1 == len);
      }
    }
    T.last_recorded = false;   // records are overwritten by the recompute of earlier segments
    for (uint32_t t = len; t-- > 0;) {
      StepRecord& r = *T.rec[t];
      DemStepView v{r.state_pos.as<double4>(), r.state_vel.as<double4>(), r.state_om.as<double4>(),
                    r.ids.as<uint32_t>(), r.perm.as<uint32_t>(), T.slot_of.as<uint32_t>(),
                    r.hcnt.as<uint32_t>(), r.hid.as<uint32_t>(), r.hxi.p, r.wxi.p,
                    (t + 1 == len ? r.hcnt_out : T.rec[t + 1]->hcnt).as<uint32_t>(),
                    (t + 1 == len ? r.hid_out : T.rec[t + 1]->hid).as<uint32_t>()};
      if (!n) continue;
      LaunchScope ls(&c, F == kF64 ? "dem_adjoint_f64" : "dem_adjoint_mixed", 0.0);
      k_dem_adj_prep<<<nb, kBlock, 0, c.stream>>>(n, c.n_moving, v, xb, vb, wb, T.cvec.as<double4>(),
                                                  T.xbf.as<double4>(), c.dem.dt, T.slot_of.as<uint32_t>());
      k_dem_adj<H><<<tile_grid(tiles), 64, 0, c.stream>>>(
          n, c.n_moving, v, kc, xb, vb, wb, T.cvec.as<double4>(), T.xbf.as<double4>(), hn, wn, mn, hp, wp, mp, xb2, vb2, wb2,
          T.partial.as<double4>() + (size_t)tiles * (len - 1u - t), tiles);
      PR_HIP(hipGetLastError());
      std::swap(xb, xb2);
      std::swap(vb, vb2);
      std::swap(wb, wb2);
      std::swap(hn, hp);
      std::swap(wn, wp);
      std::swap(mn, mp);
    }
    if (n) {   // the segment's parameter sums
      k_dem_adj_reduce<<<len, 256, 0, c.stream>>>(tiles, T.partial.as<double4>());
      PR_HIP(hipGetLastError());
      k_dem_adj_acc<<<1, 1, 0, c.stream>>>(tiles, len, T.partial.as<double4>(), T.acc.as<double>());
      PR_HIP(hipGetLastError());
    }
  }
  if (grad_params) {
    double acc[3];
    to_host(c, acc, T.acc.p, sizeof(acc));
    for (int q = 0; q < 3; ++q) grad_params[q] = acc[q];
  }
  if (grad_v0) adj_grad_scatter(c, T.ckpt[0]->ids.as<uint32_t>(), vb, grad_v0);
  restore_state(c, *T.final_state);
  c.check_flags();
}

}  // namespace prestige
