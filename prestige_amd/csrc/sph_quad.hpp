// sph_quad.hpp — the WCSPH gathers with four lanes per particle.
//
// Same passes, same sums as k_sph_density and k_sph_force; a wavefront holds
// 16 consecutive slots and each particle's four lanes (a quad) evaluate four
// neighbours at a time.  The terms are then added in list order by every lane
// of the quad (the three others' terms come through quad permutes), so each
// sum is formed in exactly the order of the one-lane kernels.
//
// Why it exists: with one lane per particle a tank of 8,000 fluid particles
// fills about 200 wavefronts of a 256-CU device, and each is a serial chain of
// nine (cell table, staging, scan, walk) rounds with a dependent gather per
// pair.  Here the nine runs' table entries are read at once, each run's
// candidates are loaded while the previous run is scanned, the hits of all
// runs become one list per particle, and the walk knows every neighbour's
// address ahead.  Density / force, us, against one lane per particle (steps
// 30-150 of a dam break): 42,866 particles FP64 63 / 44 -> 27 / 16, 196k mixed 103 /
// 51 -> 56 / 33, 571k FP32 85 / 61 -> 107 / 46.  What bounds them now: at 42,866 particles a wavefront's
// own chain (alone on its SIMD a chunk of 64 candidates takes 1,700 cycles, five
// trips through LDS and ten rounds of writing hits among them, and a round of
// the walk 1,000; deeper prefetch changes nothing); at 571k instruction issue
// and the texture path, each 80 % busy in the density pass.
#pragma once

namespace prestige {

constexpr uint32_t kQuadSlots = 16;    // particles per wavefront
constexpr uint32_t kQuadCap = 128;     // list entries per particle (LDS and nlist)
constexpr uint32_t kQuadStride = kQuadCap + 8u;   // LDS words per list: a walk row's quads read distinct banks
constexpr uint32_t kQuadRows = kQuadCap / 4u;
constexpr uint32_t kQuadOver = 0xFFFFFFFFu;   // ncnt of a tile whose lists do not fit: walked from the cell table

// Value v of lane K of the quad.
template <int K>
__device__ inline uint32_t quad_bcast(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, K * 0x55, 0xF, 0xF, true);
}
template <int K>
__device__ inline float quad_bcast(float v) {
  return __uint_as_float(quad_bcast<K>(__float_as_uint(v)));
}
template <int K>
__device__ inline double quad_bcast(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = quad_bcast<K>((uint32_t)u), hi = quad_bcast<K>((uint32_t)(u >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// fn(integral_constant K) for the quad's lanes 0..3 in order.
template <class Fn>
__device__ inline void for_quad(Fn&& fn) {
  fn(std::integral_constant<int, 0>{});
  fn(std::integral_constant<int, 1>{});
  fn(std::integral_constant<int, 2>{});
  fn(std::integral_constant<int, 3>{});
}

// Moved-slot bits of a 16-slot tile (its quarter of the mask word) from the
// quads' first lanes; every lane calls.
__device__ inline void moved_word_quad(const MovedOut& mo, uint32_t tile, bool moved) {
  uint64_t m = __ballot(moved);   // bits 4 p, packed to bits p
  m = (m | (m >> 3)) & 0x0303030303030303ull;
  m = (m | (m >> 6)) & 0x000F000F000F000Full;
  m = (m | (m >> 12)) & 0x000000FF000000FFull;
  m = (m | (m >> 24)) & 0xFFFFull;
  if (__lane_id() == 0u) reinterpret_cast<uint16_t*>(mo.mask)[tile] = (uint16_t)m;
}

// Row runs of a particle's cell in the WCSPH order: first slot and length of
// each (0 outside the grid; cut to 128 candidates, reported in over).
struct QuadRuns {
  uint32_t j0[kRuns], len[kRuns];
  bool over;
};

// First slot and length of the k-th run.
__device__ inline uint2 quad_run(const CellRows& cr, bool live, const Grid& g, const uint32_t* __restrict__ lb,
                                 uint32_t k) {
  const uint32_t r = sph_run(k);
  const int zz = cr.cz + (int)(r / 3u) - 1, yy = cr.cy + (int)(r % 3u) - 1;
  const bool ok = live && zz >= 0 && zz < g.dims[2] && yy >= 0 && yy < g.dims[1];
  const uint32_t row = ok ? ((uint32_t)zz * (uint32_t)g.dims[1] + (uint32_t)yy) * (uint32_t)g.dims[0] : 0u;
  const uint32_t a = lb[row + (uint32_t)cr.x0], b = lb[row + (uint32_t)cr.x1 + 1u];
  return make_uint2(a, ok ? b - a : 0u);
}

__device__ inline QuadRuns quad_runs(const CellRows& cr, bool live, const Grid& g, const uint32_t* __restrict__ lb) {
  QuadRuns q;
  q.over = false;
#pragma unroll
  for (uint32_t k = 0; k < kRuns; ++k) {
    const uint2 r = quad_run(cr, live, g, lb, k);
    q.j0[k] = r.x;
    q.len[k] = r.y;
  }
#pragma unroll
  for (uint32_t k = 0; k < kRuns; ++k)
    if (q.len[k] > 128u) {
      q.over = true;
      q.len[k] = 128u;
    }
  return q;
}

// Neighbours of a quad four at a time, in order, straight from the row runs
// of cell cr: fn(j, valid) with j a slot that may be read either way.
template <class Fn>
__device__ inline void quad_walk_runs(const CellRows& cr, bool live, const Grid& g, const uint32_t* __restrict__ lb,
                                      uint32_t sub, uint32_t self, Fn&& fn) {
#pragma unroll 1
  for (uint32_t k = 0; k < kRuns; ++k) {
    const uint2 q = quad_run(cr, live, g, lb, k);
    const uint32_t len = min(q.y, 128u);
    for (uint32_t b = sub; __ballot(b < len) != 0ull; b += 4u) fn(b < len ? q.x + b : self, b < len);
  }
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Hit mask of 64 candidates (the c-th in lane c's q: FP32 offsets, |q|^2 in
// .w) against the wavefront's 16 particles: lane l gets, for particle l & 15,
// bits b = 0..15 of candidates 16 (l >> 4) + b.  |s - q|^2 < t is the sign of
// q.w - 2 s.q - (t - |s|^2), a 16x4 by 4x16 product per 16 candidates: four
// FP32 matrix instructions replace 64 fused multiply-adds per lane, and each
// result costs one instruction to shift into the mask.  b: component l >> 4
// of (-2 s, 1) for particle l & 15; c: |s|^2 - t of that particle.  Row 4 h +
// v of product m holds candidate 16 h + 4 m + v, so that a lane's 16
// candidates are consecutive.  s_q: 64 float4, 16 words of padding after
// every 16 (the four row groups then read distinct banks).
__device__ inline uint32_t quad_scan64(float4* s_q, const float4& q, uint32_t lane, float b, float c) {
  s_q[lane + (lane >> 4) * 4u] = q;
  __builtin_amdgcn_wave_barrier();   // one wavefront: its LDS operations complete in order
  const float* w = reinterpret_cast<const float*>(s_q);
  const uint32_t row = lane & 15u, at = (row >> 2) * 80u + (row & 3u) * 4u + (lane >> 4);
  f32x4 d[4];
#pragma unroll
  for (uint32_t m = 0; m < 4u; ++m) {
    const f32x4 c4 = {c, c, c, c};
    d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[at + 16u * m], b, c4, 0, 0, 0);
  }
  __builtin_amdgcn_wave_barrier();
  uint32_t word = 0;
#pragma unroll
  for (int m = 3; m >= 0; --m)
#pragma unroll
    for (int v = 3; v >= 0; --v) word = __builtin_amdgcn_alignbit(word, __float_as_uint(d[m][v]), 31u);
  return word;
}

// Exclusive prefix over the four lanes l, l + 16, l + 32, l + 48 (in that
// order) and their total.
__device__ inline uint2 rows_prefix(uint32_t x, uint32_t lane) {
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);   // rows (0,0,2,2) and (1,1,3,3)
  const uint32_t pair = a[0] + a[1];
  const auto b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);   // halves
  return make_uint2(((lane & 16u) ? a[0] : 0u) + ((lane & 32u) ? b[0] : 0u), b[0] + b[1]);
}

// The four 16-bit words of lanes l, l + 16, l + 32, l + 48 as one, in that order.
__device__ inline uint64_t rows_gather16(uint32_t x) {
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const uint32_t pair = a[0] | (a[1] << 16);
  const auto b = __builtin_amdgcn_permlane32_swap(pair, pair, false, false);
  return (uint64_t)b[0] | ((uint64_t)b[1] << 32);
}

// Six wavefronts per SIMD: 500k fluid mixed 245 us a pass; with 32-bit list
// entries in LDS, which leave room for four, 281.
template <int F>
constexpr int kQuadDensWaves = 6;
// REC: the step is recorded for the adjoint, so every particle's row masks are
// stored too, in the layout of k_sph_density (42,866 particles: 27 -> 31 us).
template <int F, bool REC>
__global__ __launch_bounds__(64, kQuadDensWaves<F>) void k_sph_density_quad(
    uint32_t n, const typename SphForm<F>::S4* __restrict__ spos, const typename SphForm<F>::G4* pos,
    const uint32_t* __restrict__ skeys, const uint32_t* __restrict__ lb, Grid g, SphConst kc, SphUnits u,
    uint32_t* __restrict__ nlist, uint32_t* __restrict__ ncnt, uint2* __restrict__ meta,
    uint32_t* __restrict__ words, typename SphForm<F>::R2* __restrict__ rp, typename SphForm<F>::G4* wpos,
    typename SphForm<F>::G4* wvel, typename SphForm<F>::real* __restrict__ pres, uint32_t* flags, uint32_t n_tiles,
    DryWalls dw) {
  using real = typename SphForm<F>::real;
  using G4 = typename SphForm<F>::G4;
  using S4 = typename SphForm<F>::S4;
  __shared__ float4 s_q[80];
  __shared__ uint16_t s_l[kQuadSlots * kQuadStride];   // run << 12 | candidate of the run's union
  __shared__ uint32_t s_base[kRuns + 1u];
  const uint32_t tile = xcd_tile(blockIdx.x);
  if (tile >= n_tiles) return;
  const uint32_t lane = threadIdx.x, wbase = tile * kQuadSlots;
  // the walk: particle lane >> 2, neighbours 4 t + (lane & 3)
  const uint32_t sub = lane & 3u, p = lane >> 2, qshift = lane & ~3u;
  const uint32_t i = wbase + p;
  const bool live = i < n;
  const uint32_t self = live ? i : wbase;   // a slot every lane may read
  const G4 pi = pos[self];
  const uint32_t id = dw.ids[self];
  const bool moving = __ballot(live && (uint64_t)id < dw.n_moving) != 0ull;
  bool dry = false;
  if (dw.stamps && !moving) {
    dry = live && dry_cells(decode_cell(skeys[self], g), g, dw);
    const bool keep = !live || (dry && dw.reuse && dw.dry_pass[id] == dw.pass - 1u);
    if (dry) dw.dry_pass[id] = dw.pass;
    if (__ballot(!keep) == 0ull) {
      if constexpr (REC)
        if (live)
          for (uint32_t r = sub; r < kRuns; r += 4u) meta[meta_index(r, n, i)] = make_uint2(0u, 0u);
      if (live && sub == 0u) density_keep<F>(i, id, pi, wvel, kc, dw, rp, pres);
      return;
    }
  }
  // the scan: particle lane & 15
  const uint32_t sp = lane & 15u;
  const bool slive = wbase + sp < n;
  const uint32_t sself = slive ? wbase + sp : wbase;
  const QuadRuns qr = quad_runs(decode_cell(skeys[sself], g), slive, g, lb);
  // union of the wavefront's candidate ranges per run: slots are in key
  // order, so the first and last lane with candidates bound it
  uint32_t base[kRuns], span[kRuns];
#pragma unroll
  for (uint32_t k = 0; k < kRuns; ++k) {
    const uint32_t m = (uint32_t)__ballot(qr.len[k] != 0u) & 0xFFFFu;
    base[k] = span[k] = 0u;
    if (m != 0u) {
      const int lo = __builtin_ctz(m), hi = 31 - __builtin_clz(m);
      base[k] = (uint32_t)__builtin_amdgcn_readlane((int)qr.j0[k], lo);
      span[k] = (uint32_t)__builtin_amdgcn_readlane((int)(qr.j0[k] + qr.len[k]), hi) - base[k];
    }
  }
  const S4 p0 = spos[wbase];
  const double xr = (double)p0.x, yr = (double)p0.y, zr = (double)p0.z, ih = u.scan_inv_h;
  auto offset = [&](const S4& x) {
    float4 q = make_float4((float)(((double)x.x - xr) * ih), (float)(((double)x.y - yr) * ih),
                           (float)(((double)x.z - zr) * ih), 0.0f);
    q.w = __builtin_fmaf(q.x, q.x, __builtin_fmaf(q.y, q.y, q.z * q.z));
    return q;
  };
  const float4 so = offset(spos[sself]);
  // Rounding of the product form with |s|, |q| <= M stays below u (22 M^2 +
  // 14 M + 5), u = 2^-24 (k_sph_density), plus one rounding for the threshold
  // summed in; a candidate lies within two cells per axis of its particle, so
  // M <= |s| + 3.5 cells, and the margin is 64 u (M^2 + M + 1).
  const float M = __builtin_sqrtf(so.w) + 3.5f * u.cs_u;
  const float cneg = so.w - (u.H2_probe + 0x1.0p-18f * (M * M + M + 1.0f));
  const uint32_t h = lane >> 4;
  const float bop = h == 0u ? -2.0f * so.x : (h == 1u ? -2.0f * so.y : (h == 2u ? -2.0f * so.z : 1.0f));
  // hits of every run, in run and slot order, into the particle's list
  uint32_t scnt = 0;
  bool fits = true;
  S4 next = spos[min(base[0] + lane, n - 1u)];
#pragma unroll
  for (uint32_t k = 0; k < kRuns; ++k) {
    S4 cand = next;
    if (lane == 0u) s_base[k] = base[k];
    uint64_t m0 = 0, m1 = 0;   // REC: the run's mask, bit 0 its first candidate
    if (k + 1u < kRuns) next = spos[min(base[k + 1u] + lane, n - 1u)];
    for (uint32_t c = 0; c < span[k]; c += 64u) {
      if (c) cand = spos[min(base[k] + c + lane, n - 1u)];
      uint32_t word = quad_scan64(s_q, offset(cand), lane, bop, cneg);
      // keep the bits of the particle's own run
      const uint32_t first = base[k] + c + 16u * h;   // slot of bit 0
      const int lo = max((int)(qr.j0[k] - first), 0), hi = min((int)(qr.j0[k] + qr.len[k] - first), 16);
      word = hi > lo ? word & (((1u << (hi - lo)) - 1u) << lo) : 0u;
      if constexpr (REC) {
        const uint64_t all = rows_gather16(word);   // bit b: slot base + c + b
        const int at = (int)(base[k] + c - qr.j0[k]);   // mask bit of bit 0
        if (at <= 0) {
          if (at > -64) m0 |= all >> -at;
        } else if (at < 64) {
          m0 |= all << at;
          m1 |= all >> (64 - at);
        } else if (at < 128) {
          m1 |= all << (at - 64);
        }
      }
      const uint2 pre = rows_prefix((uint32_t)__popc(word), lane);
      fits = fits && c < 4096u && __ballot(scnt + pre.y > kQuadCap) == 0ull;
      if (fits) {
        uint16_t* l = s_l + sp * kQuadStride + scnt + pre.x;
        const uint32_t tag = (k << 12) + c + 16u * h;
        while (word) {
          *l++ = (uint16_t)(tag + (uint32_t)__builtin_ctz(word));
          word &= word - 1u;
        }
      }
      scnt += pre.y;
    }
    if constexpr (REC)
      if (slive) {
        const uint32_t r = sph_run(k);
        if (h == 0u) meta[meta_index(r, n, sself)] = make_uint2(qr.j0[k], qr.len[k]);
        const uint64_t m = h < 2u ? m0 : m1;
        if (qr.len[k] > 32u * h) words[word_index(r, h, n, sself)] = (uint32_t)((h & 1u) ? m >> 32 : m);
      }
  }
  __builtin_amdgcn_wave_barrier();
  const uint32_t cnt = __shfl(scnt, (int)p, 64);
  const real H2 = (real)u.H2, inv_h = (real)u.inv_h;
  Sum<real, F == kMixed> acc;
  // pair terms of four neighbours, then their ordered sum
  auto body = [&](const G4& pj, bool valid) {
    real dx, dy, dz, f = real(0.0);
    bool in = false;
    if constexpr (F == kMixed) quad_probe_pair(pi, pj, u.cs_u, dx, dy, dz);
    else form_pair<F>(pi, pj, u.cs_u, dx, dy, dz);
    const real r2 = dot3(dx, dy, dz, dx, dy, dz);
    if (valid && r2 < H2) {
      const real q = r2 > real(0.0) ? sqrt_pos(r2) * inv_h : real(0.0);
      f = spline_f(q);
      in = true;
    }
    if constexpr (F == kMixed) {
      const uint32_t nib = (uint32_t)(__ballot(in) >> qshift);
      for_quad([&](auto K) {
        const real t = quad_bcast<K.value>(f);
        if ((nib >> K.value) & 1u) acc.add(t);
      });
    } else {
      for_quad([&](auto K) { acc.s = acc.s + quad_bcast<K.value>(f); });   // f = 0 adds nothing
    }
  };
  if (fits) {
    uint32_t* out = nlist + (size_t)tile * (kQuadRows * 64u) + lane;
    const uint16_t* l = s_l + p * kQuadStride + sub;
    auto entry = [&](uint32_t t) {
      if (4u * t + sub >= cnt) return self;
      const uint32_t e = l[4u * t];
      return s_base[e >> 12] + (e & 4095u);
    };
    uint32_t ja = entry(0u), jb = entry(1u);
    G4 pa = pos[ja];
    for (uint32_t t = 0; __ballot(4u * t < cnt) != 0ull; ++t) {
      const uint32_t j = ja;
      const G4 pj = pa;
      ja = jb;
      pa = pos[ja];
      if (t + 2u < kQuadRows) jb = entry(t + 2u);
      if (moving) out[t * 64u] = j;
      body(pj, 4u * t + sub < cnt);
    }
  } else {
    quad_walk_runs(decode_cell(skeys[self], g), live, g, lb, sub, self,
                   [&](uint32_t j, bool valid) { body(pos[j], valid); });
  }
  if (__ballot(qr.over) != 0ull && lane == 0u) atomicOr(&flags[FLAG_CAPACITY], 1u);
  if (live && sub == 0u) {
    ncnt[i] = fits ? cnt : kQuadOver;
    density_store<F>(i, acc, kc, dry, dw, rp, wpos, wvel, pres);
  }
}

template <int F>
constexpr int kQuadForceWaves = F == kF64 ? 4 : 5;

template <int F>
__global__ __launch_bounds__(64, kQuadForceWaves<F>) void k_sph_force_quad(
    uint32_t n, uint64_t n_moving, const typename SphForm<F>::G4* __restrict__ gpos,
    const typename SphForm<F>::G4* __restrict__ gvel, const typename SphForm<F>::R2* __restrict__ rp,
    const uint32_t* __restrict__ ids, const uint32_t* __restrict__ skeys, const uint32_t* __restrict__ lb,
    const uint32_t* __restrict__ nlist, const uint32_t* __restrict__ ncnt, SphUnits u, ForceOut<F> out,
    uint32_t n_tiles) {
  using real = typename SphForm<F>::real;
  using G4 = typename SphForm<F>::G4;
  using R2 = typename SphForm<F>::R2;
  const uint32_t lane = threadIdx.x, sub = lane & 3u, p = lane >> 2, qshift = lane & ~3u;
  const uint32_t tile = xcd_tile(blockIdx.x);
  if (tile >= n_tiles) return;
  const uint32_t wbase = tile * kQuadSlots;
  const uint32_t i = wbase + p;
  const uint32_t self = i < n ? i : wbase;
  const bool live = i < n && (uint64_t)ids[self] < n_moving;
  const G4 pi = gpos[self], vi = gvel[self];
  real rhoi, pri;
  if constexpr (F == kMixed) {
    const R2 t = rp[self];
    rhoi = t.x;
    pri = t.y;
  } else {
    rhoi = pi.w;
    pri = vi.w;
  }
  const real alpha_c0 = (real)out.kc.alpha_c0, ach = alpha_c0 * (real)u.hv;
  Sum<real, F == kMixed> sx, sy, sz;
  struct Nb {
    G4 p, v;
    R2 r;
  };
  auto fetch = [&](uint32_t j) {
    Nb b;
    b.p = gpos[j];
    b.v = gvel[j];
    if constexpr (F == kMixed) b.r = rp[j];
    return b;
  };
  auto body = [&](const Nb& b, bool valid) {
    real dx, dy, dz, sc = real(0.0);
    bool in = false;
    real rhoj, prj;
    if constexpr (F == kMixed) {
      quad_probe_pair(pi, b.p, u.cs_u, dx, dy, dz);
      rhoj = b.r.x;
      prj = b.r.y;
    } else {
      form_pair<F>(pi, b.p, u.cs_u, dx, dy, dz);
      rhoj = b.p.w;
      prj = b.v.w;
    }
    if (valid) in = force_pair_sc<F>(dx, dy, dz, vi, rhoi, pri, b.v, rhoj, prj, u, ach, sc);
    if constexpr (F == kMixed) {
      const uint32_t nib = (uint32_t)(__ballot(in) >> qshift);
      for_quad([&](auto K) {
        const real s = quad_bcast<K.value>(sc), ex = quad_bcast<K.value>(dx), ey = quad_bcast<K.value>(dy),
                   ez = quad_bcast<K.value>(dz);
        if ((nib >> K.value) & 1u) {
          sx.add(s * ex);
          sy.add(s * ey);
          sz.add(s * ez);
        }
      });
    } else {
      if (!in) sc = dx = dy = dz = real(0.0);   // adds nothing below
      for_quad([&](auto K) {
        const real s = quad_bcast<K.value>(sc);
        sx.s = fmad(s, quad_bcast<K.value>(dx), sx.s);
        sy.s = fmad(s, quad_bcast<K.value>(dy), sy.s);
        sz.s = fmad(s, quad_bcast<K.value>(dz), sz.s);
      });
    }
  };
  if (__ballot(live) != 0ull) {
    const uint32_t c0 = live ? ncnt[self] : 0u;
    if (__ballot(c0 == kQuadOver) == 0ull) {
      const uint32_t* list = nlist + (size_t)tile * (kQuadRows * 64u);
      auto entry = [&](uint32_t t) { return 4u * t + sub < c0 ? list[t * 64u + lane] : self; };
      uint32_t jb = entry(0u);
      Nb a = fetch(jb);
      jb = entry(1u);
      for (uint32_t t = 0; __ballot(4u * t < c0) != 0ull; ++t) {
        const Nb b = a;
        a = fetch(jb);
        if (t + 2u < kQuadRows) jb = entry(t + 2u);
        body(b, 4u * t + sub < c0);
      }
    } else {
      quad_walk_runs(decode_cell(skeys[self], out.g), live, out.g, lb, sub, self,
                     [&](uint32_t j, bool valid) { body(fetch(j), valid); });
    }
  }
  // lane 0 of each quad integrates and writes
  const bool mine = sub == 0u && i < n;
  bool mv = false;
  if (mine) mv = force_store<F>(i, live, sx, sy, sz, out);
  moved_word_quad(out.moved, tile, mv);
}

}  // namespace prestige
