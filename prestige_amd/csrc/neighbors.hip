// neighbors.hip — cell keys, stable LSD radix sort, incremental stable sort
// between steps, reorder into key order, cell lower-bound table, id-order
// scatter/gather, and the eq1 probe.
//
// The sorted layout is what every gather kernel iterates: for a particle in
// cell (cx, cy, cz) the three cells cx-1..cx+1 of each of the nine (dy, dz)
// rows are one contiguous run [lb[row + cx-1], lb[row + cx+2]) of slots.
#include <chrono>
#include <mutex>
#include <thread>

#include "common.hpp"

namespace prestige {

// ---------------------------------------------------------------------------
// cell keys
// ---------------------------------------------------------------------------

// floor((x - lo) * inv_cs) per axis in FP64, exactly as the host oracle does;
// out-of-grid particles raise FLAG_DOMAIN and get key 0 so the sort stays in
// bounds.
__device__ inline uint32_t cell_key_of(double x, double y, double z, const Grid& g,
                                       uint32_t* flags) {
  double fx = floor((x - g.lo[0]) * g.inv_cs);
  double fy = floor((y - g.lo[1]) * g.inv_cs);
  double fz = floor((z - g.lo[2]) * g.inv_cs);
  bool ok = fx >= 0.0 && fy >= 0.0 && fz >= 0.0 && fx < (double)g.dims[0] &&
            fy < (double)g.dims[1] && fz < (double)g.dims[2];
  if (!ok) {
    atomicOr(&flags[FLAG_DOMAIN], 1u);
    return 0u;
  }
  uint32_t cx = (uint32_t)fx, cy = (uint32_t)fy, cz = (uint32_t)fz;
  return (cz * (uint32_t)g.dims[1] + cy) * (uint32_t)g.dims[0] + cx;
}

template <class T4>
__global__ __launch_bounds__(kBlock) void k_cell_keys(uint32_t n, const T4* __restrict__ pos,
                                                      Grid g, uint32_t* __restrict__ keys,
                                                      uint32_t* flags) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  T4 p = pos[i];
  keys[i] = cell_key_of((double)p.x, (double)p.y, (double)p.z, g, flags);
}

void keys_from_positions(Ctx& c) {
  c.inc_ready = false;
  if (c.n == 0) { c.keys_valid = true; return; }
  uint32_t n = (uint32_t)c.n;
  LaunchScope ls(&c, "cell_keys", 32.0 * n);
  if (c.desc.precision == PRESTIGE_F32)
    k_cell_keys<float4><<<blocks_for(n), kBlock, 0, c.stream>>>(
        n, c.pos[c.cur].as<float4>(), c.grid, c.keys[c.cur_key].as<uint32_t>(), c.flags.as<uint32_t>());
  else
    k_cell_keys<double4><<<blocks_for(n), kBlock, 0, c.stream>>>(
        n, c.pos[c.cur].as<double4>(), c.grid, c.keys[c.cur_key].as<uint32_t>(), c.flags.as<uint32_t>());
  PR_HIP(hipGetLastError());
  c.keys_valid = true;
}

// ---------------------------------------------------------------------------
// stable LSD radix sort of (key, slot) pairs, 8-bit digits
// ---------------------------------------------------------------------------
constexpr int kRadixBits = 8;
constexpr int kBuckets = 1 << kRadixBits;
constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;   // keys per thread and tile
constexpr int kTile = kSortThreads * kSortItems;
static_assert(kSortThreads == kBuckets, "one thread per bucket in the scan phases");

// Lanes of this wavefront whose digit equals mine (and whose item is valid):
// one ballot per digit bit, no shared memory.
__device__ inline uint64_t match_digit(uint32_t d, bool valid) {
  uint64_t m = __ballot(valid);
#pragma unroll
  for (int b = 0; b < kRadixBits; ++b) {
    uint64_t bal = __ballot((d >> b) & 1u);
    m &= ((d >> b) & 1u) ? bal : ~bal;
  }
  return m;
}

__device__ inline uint64_t lanes_below() {
  return (1ull << __lane_id()) - 1ull;
}

// Per-tile digit histogram: hist[d * n_tiles + tile].
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const uint32_t* __restrict__ keys,
                                                            uint32_t n, int shift,
                                                            uint32_t n_tiles,
                                                            uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[kBuckets];
  const uint32_t t = threadIdx.x;
  h[t] = 0;
  __syncthreads();
  const uint32_t base = blockIdx.x * (uint32_t)kTile;
  for (int it = 0; it < kSortItems; ++it) {
    uint32_t idx = base + (uint32_t)it * kSortThreads + t;
    bool valid = idx < n;
    uint32_t d = valid ? (keys[idx] >> shift) & (kBuckets - 1) : 0u;
    uint64_t peers = match_digit(d, valid);
    if (valid && (peers & lanes_below()) == 0ull) atomicAdd(&h[d], (uint32_t)__popcll(peers));
  }
  __syncthreads();
  hist[t * n_tiles + blockIdx.x] = h[t];
}

// Inclusive scan within a wavefront of 64 lanes.
__device__ inline uint32_t wave_incl_scan(uint32_t x) {
  const int lane = (int)__lane_id();
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    uint32_t y = __shfl_up(x, (unsigned)o, 64);
    if (lane >= o) x += y;
  }
  return x;
}

// Exclusive scan over a 256-thread block; *total receives the sum.
__device__ inline uint32_t block_excl_scan(uint32_t v, uint32_t* s4, uint32_t* total) {
  const uint32_t w = threadIdx.x >> 6;
  uint32_t x = wave_incl_scan(v);
  if (__lane_id() == 63) s4[w] = x;
  __syncthreads();
  uint32_t base = 0;
  for (uint32_t k = 0; k < w; ++k) base += s4[k];
  *total = s4[0] + s4[1] + s4[2] + s4[3];
  __syncthreads();
  return base + x - v;
}

// One block per digit: exclusive scan of hist[d][*] across tiles, tot[d] = count.
__global__ __launch_bounds__(kSortThreads) void k_sort_scan(uint32_t* __restrict__ hist,
                                                            uint32_t n_tiles,
                                                            uint32_t* __restrict__ tot) {
  __shared__ uint32_t s4[4];
  uint32_t* row = hist + (size_t)blockIdx.x * n_tiles;
  uint32_t carry = 0;
  for (uint32_t b = 0; b < n_tiles; b += kSortThreads) {
    uint32_t idx = b + threadIdx.x;
    uint32_t v = idx < n_tiles ? row[idx] : 0u;
    uint32_t total;
    uint32_t ex = block_excl_scan(v, s4, &total);
    if (idx < n_tiles) row[idx] = carry + ex;
    carry += total;
  }
  if (threadIdx.x == 0) tot[blockIdx.x] = carry;
}

// Stable scatter of one tile.  Items are taken in rounds of 256 consecutive
// slots; inside a round the rank of an item among equal digits is its
// wavefront rank (ballot match) plus the counts of earlier wavefronts, and
// rounds advance a per-digit running offset, so equal digits keep their
// input order.
__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(
    const uint32_t* __restrict__ kin, const uint32_t* __restrict__ vin, uint32_t* __restrict__ kout,
    uint32_t* __restrict__ vout, uint32_t n, int shift, uint32_t n_tiles,
    const uint32_t* __restrict__ hist, const uint32_t* __restrict__ tot) {
  __shared__ uint32_t s_run[kBuckets];
  __shared__ uint32_t s_wave[4][kBuckets];
  __shared__ uint32_t s4[4];
  const uint32_t t = threadIdx.x;
  const uint32_t w = t >> 6;
  {
    uint32_t total;
    uint32_t digit_base = block_excl_scan(tot[t], s4, &total);
    s_run[t] = digit_base + hist[t * n_tiles + blockIdx.x];
  }
  const uint32_t base = blockIdx.x * (uint32_t)kTile;
  for (int it = 0; it < kSortItems; ++it) {
    uint32_t idx = base + (uint32_t)it * kSortThreads + t;
    bool valid = idx < n;
    uint32_t k = valid ? kin[idx] : 0u;
    uint32_t v = valid ? (vin ? vin[idx] : idx) : 0u;
    uint32_t d = (k >> shift) & (kBuckets - 1);
    s_wave[0][t] = 0; s_wave[1][t] = 0; s_wave[2][t] = 0; s_wave[3][t] = 0;
    __syncthreads();
    uint64_t peers = match_digit(d, valid);
    uint32_t rank = (uint32_t)__popcll(peers & lanes_below());
    if (valid && rank == 0) s_wave[w][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    {
      uint32_t c0 = s_wave[0][t], c1 = s_wave[1][t], c2 = s_wave[2][t], c3 = s_wave[3][t];
      uint32_t r = s_run[t];
      s_wave[0][t] = r;
      s_wave[1][t] = r + c0;
      s_wave[2][t] = r + c0 + c1;
      s_wave[3][t] = r + c0 + c1 + c2;
      s_run[t] = r + c0 + c1 + c2 + c3;
    }
    __syncthreads();
    if (valid) {
      uint32_t dst = s_wave[w][d] + rank;
      kout[dst] = k;
      vout[dst] = v;
    }
    __syncthreads();
  }
}

__global__ void k_iota(uint32_t n, uint32_t* v) {
  uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = i;
}

uint64_t sort_tiles(uint64_t n) { return (n + (uint64_t)kTile - 1) / (uint64_t)kTile; }

static int key_bits(uint32_t n_cells) {
  int b = 0;
  while (b < 32 && ((uint64_t)1 << b) < (uint64_t)n_cells) ++b;
  return b;
}

// Buffers of one radix sort: key and value ping-pong pairs, the per-tile digit
// histogram (kBuckets x tiles) and the digit totals.
struct SortBufs {
  uint32_t* keys[2];
  uint32_t* vals[2];
  uint32_t* hist;
  uint32_t* tot;
};

// Sorts the n keys (< n_cells) in keys[src]; *key_out and *val_out receive
// the buffers holding the sorted keys and the permutation (sorted slot k <-
// old slot perm[k]).  c (may be null) records the launches when timing is on.
static void radix_sort_bufs(Ctx* c, const SortBufs& b, int src, uint32_t n, uint32_t n_cells, hipStream_t st,
                            int* key_out, int* val_out) {
  const int bits = key_bits(n_cells);
  const int passes = (bits + kRadixBits - 1) / kRadixBits;
  const uint32_t n_tiles = (uint32_t)sort_tiles(n);
  *key_out = src;
  *val_out = 0;
  if (passes == 0) {
    k_iota<<<blocks_for(n), kBlock, 0, st>>>(n, b.vals[0]);
    PR_HIP(hipGetLastError());
    return;
  }
  int vsrc = -1;   // first pass generates slot indices itself
  for (int p = 0; p < passes; ++p) {
    const int shift = p * kRadixBits;
    const int dst = src ^ 1;
    const int vdst = (vsrc < 0) ? 0 : (vsrc ^ 1);
    {
      LaunchScope ls(c, "sort_hist", 4.0 * n);
      k_sort_hist<<<n_tiles, kSortThreads, 0, st>>>(b.keys[src], n, shift, n_tiles, b.hist);
      PR_HIP(hipGetLastError());
    }
    {
      LaunchScope ls(c, "sort_scan", 8.0 * kBuckets * n_tiles);
      k_sort_scan<<<kBuckets, kSortThreads, 0, st>>>(b.hist, n_tiles, b.tot);
      PR_HIP(hipGetLastError());
    }
    {
      LaunchScope ls(c, "sort_scatter", (vsrc < 0 ? 12.0 : 16.0) * n);
      k_sort_scatter<<<n_tiles, kSortThreads, 0, st>>>(b.keys[src], vsrc < 0 ? nullptr : b.vals[vsrc], b.keys[dst],
                                                       b.vals[vdst], n, shift, n_tiles, b.hist, b.tot);
      PR_HIP(hipGetLastError());
    }
    src = dst;
    vsrc = vdst;
  }
  *key_out = src;
  *val_out = vsrc;
}

// Sorts keys[cur_key]; afterwards keys[cur_key] holds sorted keys and
// vals[perm_buf] the permutation (sorted slot k <- old slot perm[k]).
static void radix_sort(Ctx& c) {
  const SortBufs b{{c.keys[0].as<uint32_t>(), c.keys[1].as<uint32_t>()},
                   {c.vals[0].as<uint32_t>(), c.vals[1].as<uint32_t>()},
                   c.sort_hist.as<uint32_t>(), c.sort_tot.as<uint32_t>()};
  radix_sort_bufs(&c, b, c.cur_key, (uint32_t)c.n, c.grid.n_cells, c.stream, &c.cur_key, &c.perm_buf);
}

// ---------------------------------------------------------------------------
// reorder into key order.  PROBE also writes the FP32 probe (offset from the
// FP64 cell origin times off_scale, cell-coordinate residues mod 4 in .w);
// MIXED also writes FP32 copies of the velocity (mass in .w) and, with OMEGA,
// of the angular velocity (radius in .w).
// ---------------------------------------------------------------------------

// Gather-side copies of one particle moved from slot s to slot k (cell key
// of slot k: key): state, id, and for the mixed form the FP32 probe (offset
// from the FP64 origin of the cell, cell code in .w) and velocity copies.
template <class T4>
struct ReorderIO {
  const T4 *pos_in, *vel_in, *om_in;
  const uint32_t* id_in;
  T4 *pos_out, *vel_out, *om_out;
  uint32_t* id_out;
  Grid g;
  float4 *off32, *vel32, *om32;
};

template <class T4, bool OMEGA, bool PROBE, bool MIXED>
__device__ inline void move_slot(const ReorderIO<T4>& io, uint32_t s, uint32_t k, uint32_t key) {
  const T4 p = io.pos_in[s];
  const T4 v = io.vel_in[s];
  io.pos_out[k] = p;
  io.vel_out[k] = v;
  io.id_out[k] = io.id_in[s];
  if constexpr (OMEGA) {
    const T4 w = io.om_in[s];
    io.om_out[k] = w;
    if constexpr (MIXED) io.om32[k] = make_float4((float)w.x, (float)w.y, (float)w.z, (float)p.w);
  }
  if constexpr (PROBE) {
    const Grid& g = io.g;
    const uint32_t cx = key % (uint32_t)g.dims[0];
    const uint32_t rest = key / (uint32_t)g.dims[0];
    const uint32_t cy = rest % (uint32_t)g.dims[1];
    const uint32_t cz = rest / (uint32_t)g.dims[1];
    const float ox = (float)(((double)p.x - (g.lo[0] + (double)cx * g.cs)) * g.off_scale);
    const float oy = (float)(((double)p.y - (g.lo[1] + (double)cy * g.cs)) * g.off_scale);
    const float oz = (float)(((double)p.z - (g.lo[2] + (double)cz * g.cs)) * g.off_scale);
    io.off32[k] = make_float4(ox, oy, oz, __uint_as_float(cell_code(cx, cy, cz)));
  }
  if constexpr (MIXED) io.vel32[k] = make_float4((float)v.x, (float)v.y, (float)v.z, (float)v.w);
}

template <class T4, bool OMEGA, bool PROBE, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_reorder(uint32_t n, const uint32_t* __restrict__ perm,
                                                    const uint32_t* __restrict__ skeys, ReorderIO<T4> io) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) move_slot<T4, OMEGA, PROBE, MIXED>(io, perm[k], k, skeys[k]);
}

// The copies of one build from buffer src to dst, as the context's model and
// precision need them.
template <class T4, bool OMEGA, bool MIXED>
ReorderIO<T4> reorder_io(Ctx& c, int src, int dst) {
  return ReorderIO<T4>{c.pos[src].as<T4>(), c.vel[src].as<T4>(), OMEGA ? c.omega[src].as<T4>() : nullptr,
                       c.ids[c.cur_ids].as<uint32_t>(), c.pos[dst].as<T4>(), c.vel[dst].as<T4>(),
                       OMEGA ? c.omega[dst].as<T4>() : nullptr, c.ids[c.cur_ids ^ 1].as<uint32_t>(), c.grid,
                       MIXED ? c.off32.as<float4>() : nullptr, MIXED ? c.vel32.as<float4>() : nullptr,
                       (MIXED && OMEGA) ? c.om32.as<float4>() : nullptr};
}

// The copy variant as a type: fn(ReorderForm<...>{}, io) picks the kernel.
template <class T4, bool OMEGA, bool PROBE, bool MIXED>
struct ReorderForm {
  using T = T4;
  static constexpr bool omega = OMEGA, probe = PROBE, mixed = MIXED;
};

// Calls fn(form, io) for the context's form (the mixed forms build the FP32
// probe; DEM moves omega).
template <class Fn>
void with_reorder_form(Ctx& c, int src, int dst, Fn&& fn) {
  const bool dem = c.desc.model == PRESTIGE_MODEL_DEM;
  const bool sph = c.desc.model == PRESTIGE_MODEL_WCSPH;
  const bool mixed = c.desc.precision == PRESTIGE_MIXED;
  const bool f32 = c.desc.precision == PRESTIGE_F32;
  if (dem) {
    if (mixed) fn(ReorderForm<double4, true, true, true>{}, reorder_io<double4, true, true>(c, src, dst));
    else fn(ReorderForm<double4, true, false, false>{}, reorder_io<double4, true, false>(c, src, dst));
  } else if (f32) {
    fn(ReorderForm<float4, false, false, false>{}, reorder_io<float4, false, false>(c, src, dst));
  } else if (sph && mixed) {
    fn(ReorderForm<double4, false, true, true>{}, reorder_io<double4, false, true>(c, src, dst));
  } else {
    fn(ReorderForm<double4, false, false, false>{}, reorder_io<double4, false, false>(c, src, dst));
  }
}

// Bytes one build moves per particle in the reorder.
double reorder_bytes(const Ctx& c) {
  const bool dem = c.desc.model == PRESTIGE_MODEL_DEM;
  const bool mixed = c.desc.precision == PRESTIGE_MIXED;
  const bool f32 = c.desc.precision == PRESTIGE_F32;
  const double elem = f32 ? 12.0 : 24.0;   // three coordinates per vector
  return 4.0 + 2.0 * (2.0 * elem + 4.0) + (dem ? 2.0 * elem + 16.0 : 0.0) + (mixed ? 4.0 + 16.0 + 16.0 : 0.0) +
         (mixed && dem ? 16.0 : 0.0);
}

// ---------------------------------------------------------------------------
// incremental stable sort.  Between two builds only the slots whose particle
// changed cell ("moved") break the order: slots are in key_old order, and the
// kept slots of a cell keep their relative order.  The stable sort puts into
// cell c, in this order, the slots that moved in from lower cells, the kept
// ones and those from higher cells, each by slot (old slot order is old key
// order), so with the new cell table lb and the list of c's incoming slots
//   kept slot i:               lb[c] + #{incoming < i} + i - lb_old[c]
//                                - #{moved slots in [lb_old[c], i)}
//   incoming, i < lb_old[c]:   lb[c] + #{incoming < i}
//   incoming, i >= lb_old[c+1]: lb[c+1] - #{incoming >= i}
// and lb[c] is lb_old[c] plus the prefix of (in - out) over the cells before
// c.  The step kernel counted and listed the moved slots (MovedOut), so two
// launches, the cell table and the placement, which also moves the particle
// state, replace the radix sort's launches, the reorder and the cell table's;
// permutation and keys are exactly the stable sort's.  Lists have no order (the
// step's atomics link them), but only counts are taken from them.  Small scenes
// do both in one launch (k_inc_one).
//
// Us per step, against gathering the moved entries, sorting them, merging and
// a cell table (up to 8,192 moved; the radix path above): 42,866 particles 19
// -> 11, 10,000 spheres 14 -> 9, 1.8M mixed 95 -> 66, 6M FP64 (about 20,000
// moved a step) 334 -> 181.  The table costs 8 bytes a cell, the placement is
// bound by the state it moves (6 TB/s at 6M).
// ---------------------------------------------------------------------------

// New cell table of tile b (kCellTile cells): the offset before it, from the nets
// of the tile groups before its own (net; none where there is one group) and the
// totals of the tiles before it in its group, then a block scan of the cells' net
// counts, which are cleared for the next step.  A tile nothing entered or left only
// adds its offset.  (With the totals of every tile before it a step of 20,000
// spheres took 1,586 us in 101M cells and 8,032 in 238M; so 260 and 583.)
template <bool CLEAR>
__device__ inline void cell_tile(uint32_t b, uint32_t n_cells, const uint32_t* __restrict__ lb_old,
                                 const uint32_t* __restrict__ net, const uint32_t* __restrict__ tin,
                                 const uint32_t* __restrict__ tout,
                                 uint4* __restrict__ cin, uint4* __restrict__ cout, uint32_t* __restrict__ lb) {
  static_assert(kCellTile == 4 * kBlock, "four cells per thread");
  __shared__ uint32_t s4[4];
  const uint32_t t = threadIdx.x;
  const bool busy = (tin[b] | tout[b]) != 0u;
  uint32_t part = 0;
  for (uint32_t k = t; k < b / kTileGroup; k += kBlock) part += net[k];
  static_assert(kTileGroup == (uint32_t)kBlock, "one tile of the group per thread");
  if (t < b % kTileGroup) part += tin[b / kTileGroup * kTileGroup + t] - tout[b / kTileGroup * kTileGroup + t];
  part = wave_sum(part);
  if (__lane_id() == 0) s4[t >> 6] = part;
  __syncthreads();
  uint32_t run = s4[0] + s4[1] + s4[2] + s4[3];
  uint32_t d[4] = {0u, 0u, 0u, 0u};
  if (busy) {
    __syncthreads();
    const uint32_t q = b * kBlock + t;
    const uint4 in = cin[q], out = cout[q];
    d[0] = in.x - out.x; d[1] = in.y - out.y; d[2] = in.z - out.z; d[3] = in.w - out.w;
    if (CLEAR && (in.x | in.y | in.z | in.w)) cin[q] = make_uint4(0u, 0u, 0u, 0u);
    if (CLEAR && (out.x | out.y | out.z | out.w)) cout[q] = make_uint4(0u, 0u, 0u, 0u);
    uint32_t total;
    run += block_excl_scan(d[0] + d[1] + d[2] + d[3], s4, &total);
  }
  const uint32_t c0 = b * kCellTile + 4u * t;
#pragma unroll
  for (uint32_t k = 0; k < 4u; ++k) {
    if (c0 + k <= n_cells) lb[c0 + k] = lb_old[c0 + k] + run;
    run += d[k];
  }
}

__global__ __launch_bounds__(kBlock) void k_inc_cells(uint32_t n_cells, const uint32_t* __restrict__ lb_old,
                                                      const uint32_t* __restrict__ net,
                                                      const uint32_t* __restrict__ tin,
                                                      const uint32_t* __restrict__ tout, uint4* __restrict__ cin,
                                                      uint4* __restrict__ cout, uint32_t* __restrict__ lb) {
  cell_tile<true>(blockIdx.x, n_cells, lb_old, net, tin, tout, cin, cout, lb);
}

// Set bits of the moved-slot mask in [a, b).
__device__ inline uint32_t moved_in(const uint64_t* __restrict__ mask, uint32_t a, uint32_t b) {
  if (a >= b) return 0u;
  const uint32_t wa = a >> 6, wb = (b - 1u) >> 6;
  uint64_t w = mask[wa] & (~0ull << (a & 63u));
  uint32_t cnt = 0;
  for (uint32_t k = wa; k < wb; w = mask[++k]) cnt += (uint32_t)__popcll(w);
  const uint32_t top = b & 63u;   // 0: the last word counts whole
  return cnt + (uint32_t)__popcll(top ? w & ((1ull << top) - 1ull) : w);
}

// Place in the new order of slot i, now in cell c: o0, o1 and l0, l1 are the
// cell's bounds in the old and the new table, hd its list's head.
__device__ inline uint32_t place_of(uint32_t i, uint32_t o0, uint32_t o1, uint32_t l0, uint32_t l1, uint64_t hd,
                                    uint32_t epoch, const uint64_t* __restrict__ mask,
                                    const uint32_t* __restrict__ next) {
  uint32_t below = 0, above = 0;   // incoming slots before i, and i or after it
  if ((uint32_t)(hd >> 32) == epoch)
    for (uint32_t e = (uint32_t)hd; e != kListEnd; e = next[e]) {
      below += e < i ? 1u : 0u;
      above += e < i ? 0u : 1u;
    }
  if (i < o0) return l0 + below;
  if (i >= o1) return l1 - above;
  return l0 + below + (i - o0) - moved_in(mask, o0, i);
}

// One thread per slot: its place in the new order; key, permutation and the
// particle's state go there.  Also clears the tile totals and their groups' nets.
template <class T4, bool OMEGA, bool PROBE, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_inc_place(
    uint32_t n, uint32_t cell_tiles, const uint32_t* __restrict__ knew, const uint64_t* __restrict__ mask,
    const uint64_t* __restrict__ head, const uint32_t* __restrict__ next, uint32_t epoch,
    const uint32_t* __restrict__ lb_old, const uint32_t* __restrict__ lb, uint32_t* __restrict__ net,
    uint32_t* __restrict__ tin, uint32_t* __restrict__ tout, uint32_t* __restrict__ kout, uint32_t* __restrict__ perm,
    ReorderIO<T4> io) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  for (uint32_t k = i; k < cell_tiles; k += gridDim.x * (uint32_t)kBlock) {
    tin[k] = tout[k] = 0u;
    if (k % kTileGroup == 0u) net[k / kTileGroup] = 0u;
  }
  if (i >= n) return;
  const uint32_t c = knew[i];
  const uint32_t pos = place_of(i, lb_old[c], lb_old[c + 1u], lb[c], lb[c + 1u], head[c], epoch, mask, next);
  if (pos >= n) return;   // never, when the counts are consistent
  kout[pos] = c;
  perm[pos] = i;
  move_slot<T4, OMEGA, PROBE, MIXED>(io, i, pos, c);
}

// Both in one launch, for small scenes, whose builds are bound by launches and
// chains of dependent loads (two of 6-7 us; one of 7-9): the first place_blocks blocks place, each slot taking its cell's new
// bounds from the counts themselves (the tiles before, scanned by the block;
// the tile's groups before; the group's cells before: 24 independent loads that
// neighbouring slots share), the others write the table.  Nothing here may be
// cleared while another block reads it, so the table's blocks clear the set of
// counts that the build before this one read.
struct IncSet {
  uint4 *cin, *cout, *net;
  uint32_t *tin, *tout;
};
// Elements first, first + 1, ... of v whose number is below end, added up.
__device__ inline uint32_t sum_below(uint4 v, uint32_t first, uint32_t end) {
  return (first < end ? v.x : 0u) + (first + 1u < end ? v.y : 0u) + (first + 2u < end ? v.z : 0u) +
         (first + 3u < end ? v.w : 0u);
}
template <class T4, bool OMEGA, bool PROBE, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_inc_one(
    uint32_t n, uint32_t n_cells, uint32_t cell_tiles, uint32_t place_blocks, const uint32_t* __restrict__ knew,
    const uint64_t* __restrict__ mask, const uint64_t* __restrict__ head, const uint32_t* __restrict__ next,
    uint32_t epoch, const uint32_t* __restrict__ lb_old, uint32_t* __restrict__ lb, IncSet in, IncSet old,
    uint32_t* __restrict__ kout, uint32_t* __restrict__ perm, ReorderIO<T4> io) {
  constexpr uint32_t kGroups = kCellTile / kCellGroup;
  const uint32_t t = threadIdx.x;
  if (blockIdx.x >= place_blocks) {
    const uint32_t b = blockIdx.x - place_blocks;
    cell_tile<false>(b, n_cells, lb_old, nullptr, in.tin, in.tout, in.cin, in.cout, lb);
    const bool stale = (old.tin[b] | old.tout[b]) != 0u;
    __syncthreads();
    if (!stale) return;
    old.cin[b * kBlock + t] = old.cout[b * kBlock + t] = make_uint4(0u, 0u, 0u, 0u);
    if (t < kGroups / 4u) old.net[b * (kGroups / 4u) + t] = make_uint4(0u, 0u, 0u, 0u);
    if (t == 0u) old.tin[b] = old.tout[b] = 0u;
    return;
  }
  __shared__ uint32_t s4[4], s_off[kBlock];
  __shared__ bool s_busy[kBlock];
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + t;
  const uint32_t c = i < n ? knew[i] : 0u;
  const uint32_t ti = t < cell_tiles ? in.tin[t] : 0u, to = t < cell_tiles ? in.tout[t] : 0u;
  const uint32_t o0 = lb_old[c], o1 = lb_old[c + 1u];
  const uint64_t hd = head[c];
  uint32_t total;
  s_off[t] = block_excl_scan(ti - to, s4, &total);
  s_busy[t] = (ti | to) != 0u;
  __syncthreads();
  if (i >= n) return;
  const uint32_t b = c / kCellTile;
  uint32_t before = s_off[b], upto = before;   // what the cell's bounds move by
  if (s_busy[b]) {
    const uint4* __restrict__ g = in.net + b * (kGroups / 4u);
    const uint32_t q = c / kCellGroup * (kCellGroup / 4u);
    uint4 vg[kGroups / 4u], vi[kCellGroup / 4u], vo[kCellGroup / 4u];
#pragma unroll
    for (uint32_t k = 0; k < kGroups / 4u; ++k) vg[k] = g[k];
#pragma unroll
    for (uint32_t k = 0; k < kCellGroup / 4u; ++k) { vi[k] = in.cin[q + k]; vo[k] = in.cout[q + k]; }
    const uint32_t ng = c / kCellGroup % kGroups, nc = c % kCellGroup;
#pragma unroll
    for (uint32_t k = 0; k < kGroups / 4u; ++k) before += sum_below(vg[k], 4u * k, ng);
    upto = before;
#pragma unroll
    for (uint32_t k = 0; k < kCellGroup / 4u; ++k) {
      const uint4 d = make_uint4(vi[k].x - vo[k].x, vi[k].y - vo[k].y, vi[k].z - vo[k].z, vi[k].w - vo[k].w);
      before += sum_below(d, 4u * k, nc);
      upto += sum_below(d, 4u * k, nc + 1u);
    }
  }
  const uint32_t pos = place_of(i, o0, o1, o0 + before, o1 + upto, hd, epoch, mask, next);
  if (pos >= n) return;   // never, when the counts are consistent
  kout[pos] = c;
  perm[pos] = i;
  move_slot<T4, OMEGA, PROBE, MIXED>(io, i, pos, c);
}

// One launch pays while a launch weighs more than the extra loads of every
// slot.  Us a step, two launches / one: spheres 1,000 17.2 / 14.2, 10,000 19.8 /
// 17.3, 100,000 42.0 / 39.5; slots of a dam break, 42,866 49.1 / 47.1, 196k mixed
// 95.0 / 92.8, 329k 132.3 / 130.8, 664k F32 183.3 / 183.9.  A block scans the
// tiles with a thread each, so there may be no more of them.
constexpr uint64_t kIncOne = 400000;
bool inc_in_one(uint64_t n, size_t cell_tiles) { return cell_tiles <= (size_t)kBlock && n <= kIncOne; }

MovedOut moved_out(Ctx& c) {
  if (!c.inc_fits()) {
    MovedOut mo{};
    mo.mask = c.inc_mask.as<uint64_t>();
    return mo;
  }
  c.inc_counts = true;
  const int s = c.inc_set;
  if (++c.inc_epoch == 0u) {   // wrapped: heads left 2^32 steps ago, or never written, would pass for this step's
    PR_HIP(hipMemsetAsync(c.inc_head(), 0, c.inc_head_bytes(), c.stream));
    c.inc_epoch = 1u;
  }
  return MovedOut{c.inc_mask.as<uint64_t>(), c.inc_cin(s), c.inc_cout(s), c.inc_tin(s), c.inc_tout(s), c.inc_net(s),
                  c.inc_head(), c.inc_next.as<uint32_t>(), c.inc_epoch, c.inc_net_shift()};
}

static void inc_taken(Ctx& c) {
  std::swap(c.lb.p, c.lb_spare.p);
  c.inc_counts = false;
  c.cur_key ^= 1;
  c.perm_buf = 0;
}

// Stable sort of keys[cur_key] from the previous build's order (keys[cur_key
// ^ 1] = its sorted keys, lb its cell table), with the new cell table and the
// state moved; same outputs as radix_sort, k_reorder and k_cell_lb.
static void incremental_sort(Ctx& c) {
  const uint32_t n = (uint32_t)c.n;
  const uint32_t cells = c.grid.n_cells;
  const uint32_t tiles = (uint32_t)c.inc_tiles;
  if (c.inc_one) {
    LaunchScope ls(&c, "sort_inc_one", 8.0 * cells + (12.0 + reorder_bytes(c)) * n);
    auto set = [&](int s) {
      return IncSet{reinterpret_cast<uint4*>(c.inc_cin(s)), reinterpret_cast<uint4*>(c.inc_cout(s)),
                    reinterpret_cast<uint4*>(c.inc_net(s)), c.inc_tin(s), c.inc_tout(s)};
    };
    with_reorder_form(c, c.cur, c.cur ^ 1, [&](auto form, auto io) {
      using F = decltype(form);
      const uint32_t place_blocks = blocks_for(n);
      k_inc_one<typename F::T, F::omega, F::probe, F::mixed><<<place_blocks + tiles, kBlock, 0, c.stream>>>(
          n, cells, tiles, place_blocks, c.keys[c.cur_key].as<uint32_t>(), c.inc_mask.as<uint64_t>(), c.inc_head(),
          c.inc_next.as<uint32_t>(), c.inc_epoch, c.lb.as<uint32_t>(), c.lb_spare.as<uint32_t>(), set(c.inc_set),
          set(c.inc_set ^ 1), c.keys[c.cur_key ^ 1].as<uint32_t>(), c.vals[0].as<uint32_t>(), io);
    });
    PR_HIP(hipGetLastError());
    c.inc_set ^= 1;
    return inc_taken(c);
  }
  {
    LaunchScope ls(&c, "sort_inc_cells", 8.0 * cells);
    k_inc_cells<<<tiles, kBlock, 0, c.stream>>>(cells, c.lb.as<uint32_t>(), c.inc_net(0), c.inc_tin(0), c.inc_tout(0),
                                                reinterpret_cast<uint4*>(c.inc_cin(0)),
                                                reinterpret_cast<uint4*>(c.inc_cout(0)), c.lb_spare.as<uint32_t>());
    PR_HIP(hipGetLastError());
  }
  {
    LaunchScope ls(&c, "sort_inc_place", (12.0 + reorder_bytes(c)) * n);
    with_reorder_form(c, c.cur, c.cur ^ 1, [&](auto form, auto io) {
      using F = decltype(form);
      k_inc_place<typename F::T, F::omega, F::probe, F::mixed><<<blocks_for(n), kBlock, 0, c.stream>>>(
          n, tiles, c.keys[c.cur_key].as<uint32_t>(), c.inc_mask.as<uint64_t>(), c.inc_head(),
          c.inc_next.as<uint32_t>(), c.inc_epoch, c.lb.as<uint32_t>(), c.lb_spare.as<uint32_t>(), c.inc_net(0),
          c.inc_tin(0), c.inc_tout(0), c.keys[c.cur_key ^ 1].as<uint32_t>(), c.vals[0].as<uint32_t>(), io);
    });
    PR_HIP(hipGetLastError());
  }
  inc_taken(c);
}

// ---------------------------------------------------------------------------
// counting sort: the first build of a state, and eq1 without allocating
// ---------------------------------------------------------------------------
// Every slot takes a number within its cell as it arrives, a scan of the cell
// counts is the cell table, and the cell lists that follow from both give each
// slot its place: the start of its cell plus the slots of the cell before it
// (a stable sort, whatever the order of arrival).  The placement moves the
// state, so keys, permutation, cell table and sorted state are those of the
// radix sort with its reorder and cell table, in six launches for its eleven
// (three digits).  Us: 1M scattered points 146 -> 93, 571k particles in tank
// order 83 -> 35, 1,000 in 1,000 cells 60 -> 32.
//
// The radix sort keeps what does not pay here.  The table costs 16 bytes a
// cell: 4.1M cells with 300k particles 110 -> 59, but with 20k 107 either way, so
// the line lies at kCountCells.  A slot reads its cell's whole list: 3,000
// particles in one cell take 92 us and 106 by radix, 20,000 344 and 113, a million
// 110,000 and 160 (a particle outside the grid counts into cell 0, so that wrong
// units put all of them there).  So a context's build turns back at a cell of more
// than kCountMost, which the host hears of while the table and the lists are
// written, and sorts by radix: 20,000 in 110, a million in 240.  Asking costs the
// builds that go on up to 4 us.  eq1 without allocating does not ask, being quadratic
// in a crowd itself.
constexpr uint32_t kCountCells = 1u << 22;
constexpr uint32_t kCountMost = 2048;

static bool count_sort_fits(uint32_t n, uint32_t n_cells) {
  if ((uint64_t)n > (uint64_t)kCountMost * n_cells) return false;   // some cell has more
  // the tile totals live in the radix sort's histogram
  const uint64_t tiles = ((uint64_t)n_cells + 1u + kCellTile - 1u) / kCellTile;
  return n_cells <= kCountCells && tiles <= (uint64_t)kBuckets * sort_tiles(n);
}

// Also clears the first n_words of words.
__global__ __launch_bounds__(kBlock) void k_count_clear(uint32_t n, uint32_t* __restrict__ cnt, uint32_t n_words,
                                                        uint32_t* __restrict__ words) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (i < n) cnt[i] = 0u;
  if (i < n_words) words[i] = 0u;
}

// A device word that the count of a cell sets when it passes kCountMost; the counting
// sort's kernels may then leave their outputs unwritten.  The kernel after the counts
// tells the host: note is 2 build + (the word).
struct Crowd {
  uint32_t *word, *note;
  uint32_t build;
  __device__ bool seen() const { return __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u; }
  __device__ void set() const { __hip_atomic_store(word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ void tell() const {
    __hip_atomic_store(note, 2u * build + (seen() ? 1u : 0u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
};

// This lane's number in cell key; the lanes of a wavefront that follow each
// other into one cell take theirs with one atomic (571k particles in tank order:
// 40 -> 4.5 us; points in no order find nothing to share).  All lanes call.
// crowd may be null.
__device__ inline uint32_t cell_arrival(uint32_t* __restrict__ cnt, uint32_t key, bool live, const Crowd* crowd) {
  const uint32_t lane = __lane_id();
  const uint32_t before = (uint32_t)__shfl_up((int)key, 1, 64);
  const uint64_t starts = __ballot(lane == 0u || key != before || !live);
  const uint32_t first = 63u - (uint32_t)__builtin_clzll(starts & (~0ull >> (63u - lane)));
  const uint64_t after = lane == 63u ? 0ull : starts & (~0ull << (lane + 1u));
  const uint32_t end = after ? (uint32_t)__builtin_ctzll(after) : 64u;
  uint32_t base = 0;
  if (live && first == lane) {
    base = atomicAdd(&cnt[key], end - first);
    if (crowd && base <= kCountMost && base + (end - first) > kCountMost) crowd->set();
  }
  return (uint32_t)__shfl((int)base, (int)first, 64) + lane - first;
}

__global__ __launch_bounds__(kBlock) void k_count_keys(uint32_t n, const uint32_t* __restrict__ keys,
                                                       uint32_t* __restrict__ cnt, uint32_t* __restrict__ arr,
                                                       Crowd crowd) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  const bool live = i < n;
  const uint32_t key = live ? keys[i] : 0u;
  if (crowd.seen()) return;   // a million atomics on one count would take longer than the radix sort
  const uint32_t a = cell_arrival(cnt, key, live, &crowd);
  if (live) arr[i] = a;
}

__global__ __launch_bounds__(kBlock) void k_count_tiles(uint32_t n_cells, const uint32_t* __restrict__ cnt,
                                                        uint32_t* __restrict__ tot, Crowd crowd) {
  __shared__ uint32_t s4[4];
  if (crowd.note && blockIdx.x == 0u && threadIdx.x == 0u) crowd.tell();
  uint32_t sum = 0;
#pragma unroll
  for (uint32_t k = 0; k < kCellTile / kBlock; ++k) {
    const uint32_t c = blockIdx.x * kCellTile + k * kBlock + threadIdx.x;
    if (c < n_cells) sum += cnt[c];
  }
  sum = wave_sum(sum);
  if (__lane_id() == 0) s4[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) tot[blockIdx.x] = s4[0] + s4[1] + s4[2] + s4[3];
}

// Counts to cell table, in place.
__global__ __launch_bounds__(kBlock) void k_count_table(uint32_t n_cells, const uint32_t* __restrict__ tot,
                                                        uint32_t* __restrict__ lb) {
  __shared__ uint32_t s4[4];
  const uint32_t b = blockIdx.x, t = threadIdx.x;
  uint32_t part = 0;
  for (uint32_t k = t; k < b; k += kBlock) part += tot[k];
  part = wave_sum(part);
  if (__lane_id() == 0) s4[t >> 6] = part;
  __syncthreads();
  uint32_t run = s4[0] + s4[1] + s4[2] + s4[3];
  __syncthreads();
  const uint32_t c0 = b * kCellTile + 4u * t;
  uint32_t d[4];
#pragma unroll
  for (uint32_t k = 0; k < 4u; ++k) d[k] = c0 + k < n_cells ? lb[c0 + k] : 0u;
  uint32_t total;
  run += block_excl_scan(d[0] + d[1] + d[2] + d[3], s4, &total);
#pragma unroll
  for (uint32_t k = 0; k < 4u; ++k) {
    if (c0 + k <= n_cells) lb[c0 + k] = run;
    run += d[k];
  }
}

__global__ __launch_bounds__(kBlock) void k_count_list(uint32_t n, const uint32_t* __restrict__ keys,
                                                       const uint32_t* __restrict__ arr,
                                                       const uint32_t* __restrict__ lb, uint32_t* __restrict__ list,
                                                       Crowd crowd) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (crowd.seen()) return;   // arr is not complete
  if (i < n) list[lb[keys[i]] + arr[i]] = i;
}

// Place of slot i of a cell with entries [l0, l1) of the lists: l0 plus the
// entries below i.  A crowded cell is read 128 bytes at a time (20,000 slots in
// one cell: 620 -> 310 us, of the 5,700 that eq1 then takes over them).
__device__ inline uint32_t place_in_cell(const uint32_t* __restrict__ list, uint32_t l0, uint32_t l1, uint32_t i) {
  uint32_t pos = l0, q = l0;
  if (l1 - l0 > 64u) {
    for (; q & 3u; ++q) pos += list[q] < i ? 1u : 0u;
    const uint4* l4 = reinterpret_cast<const uint4*>(list);
    for (; q + 32u <= l1; q += 32u) {
      uint4 v[8];
#pragma unroll
      for (uint32_t k = 0; k < 8u; ++k) v[k] = l4[(q >> 2) + k];
#pragma unroll
      for (uint32_t k = 0; k < 8u; ++k)
        pos += (v[k].x < i ? 1u : 0u) + (v[k].y < i ? 1u : 0u) + (v[k].z < i ? 1u : 0u) + (v[k].w < i ? 1u : 0u);
    }
  }
#pragma unroll 4
  for (; q < l1; ++q) pos += list[q] < i ? 1u : 0u;
  return pos;
}

template <class T4, bool OMEGA, bool PROBE, bool MIXED>
__global__ __launch_bounds__(kBlock) void k_count_place(uint32_t n, const uint32_t* __restrict__ keys,
                                                        const uint32_t* __restrict__ lb,
                                                        const uint32_t* __restrict__ list,
                                                        uint32_t* __restrict__ skeys, uint32_t* __restrict__ perm,
                                                        ReorderIO<T4> io) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t c = keys[i];
  const uint32_t pos = place_in_cell(list, lb[c], lb[c + 1u], i);
  skeys[pos] = c;
  perm[pos] = i;
  move_slot<T4, OMEGA, PROBE, MIXED>(io, i, pos, c);
}

// n_cells + 1 counts (the last unused) to the cell table; tot: a total per tile;
// crowd.note may be null.
static void count_table(Ctx* c, uint32_t n_cells, uint32_t* cnt, uint32_t* tot, const Crowd& crowd, hipStream_t st) {
  LaunchScope ls(c, "sort_count_cells", 12.0 * n_cells);
  const uint32_t tiles = blocks_for((uint64_t)n_cells + 1u, (int)kCellTile);
  k_count_tiles<<<tiles, kBlock, 0, st>>>(n_cells, cnt, tot, crowd);
  PR_HIP(hipGetLastError());
  k_count_table<<<tiles, kBlock, 0, st>>>(n_cells, tot, cnt);
  PR_HIP(hipGetLastError());
}

// The counting sort of keys[cur_key] with the state moved; same outputs as
// radix_sort, k_reorder and k_cell_lb.  False, with keys[cur_key] and the state as
// they were, when a cell has more than kCountMost slots.
static bool context_count_sort(Ctx& c) {
  const uint32_t n = (uint32_t)c.n, cells = c.grid.n_cells;
  const uint32_t* keys = c.keys[c.cur_key].as<uint32_t>();
  uint32_t* arr = c.vals[0].as<uint32_t>();
  const bool ask = n > kCountMost;
  const uint32_t build = ask ? ++c.count_builds & 0x7FFFFFFFu : 0u;
  const Crowd crowd{c.flags.as<uint32_t>() + FLAG_COUNT + 1, ask ? c.note_dev + kNoteCrowd : nullptr, build};
  {
    LaunchScope ls(&c, "sort_count", 4.0 * cells + 12.0 * n);
    k_count_clear<<<blocks_for(cells + 1u), kBlock, 0, c.stream>>>(cells + 1u, c.lb.as<uint32_t>(), 1u, crowd.word);
    PR_HIP(hipGetLastError());
    k_count_keys<<<blocks_for(n), kBlock, 0, c.stream>>>(n, keys, c.lb.as<uint32_t>(), arr, crowd);
    PR_HIP(hipGetLastError());
  }
  count_table(&c, cells, c.lb.as<uint32_t>(), c.sort_hist.as<uint32_t>(), crowd, c.stream);
  uint32_t* list = c.vals[1].as<uint32_t>();
  {
    LaunchScope ls(&c, "sort_count_list", 16.0 * n);
    k_count_list<<<blocks_for(n), kBlock, 0, c.stream>>>(n, keys, arr, c.lb.as<uint32_t>(), list, crowd);
    PR_HIP(hipGetLastError());
  }
  if (ask) {
    // A wait for an event leaves the device idle twice as long (in the segments of an
    // adjoint sweep, where the host is a millisecond ahead, 15 us against 5); a wait
    // of more than 2 ms is left to the runtime.
    volatile const uint32_t* told = c.note + kNoteCrowd;
    const auto from = std::chrono::steady_clock::now();
    while (*told >> 1 != build && std::chrono::steady_clock::now() - from < std::chrono::milliseconds(2))
      std::this_thread::yield();
    if (*told >> 1 != build) PR_HIP(hipStreamSynchronize(c.stream));
    if (*told & 1u) return false;
  }
  LaunchScope ls(&c, "sort_count_place", (8.0 + reorder_bytes(c)) * n);
  with_reorder_form(c, c.cur, c.cur ^ 1, [&](auto form, auto io) {
    using F = decltype(form);
    k_count_place<typename F::T, F::omega, F::probe, F::mixed><<<blocks_for(n), kBlock, 0, c.stream>>>(
        n, keys, c.lb.as<uint32_t>(), list, c.keys[c.cur_key ^ 1].as<uint32_t>(), arr, io);
  });
  PR_HIP(hipGetLastError());
  c.cur_key ^= 1;
  c.perm_buf = 0;
  return true;
}

// lb[c] = first slot with key >= c, for c = 0 .. n_cells.  Thread k < n owns
// the cells [lo, hi) whose lower bound is k: lo = key[k-1] + 1 (0 for k = 0),
// hi = key[k] + 1; the cells after the last key (lower bound n: the empty
// top of the domain) are spread over kTailBlocks extra blocks.  Every cell
// is written exactly once and no clearing pass is needed.  A lane writes a
// range of up to kOwnCells cells itself; longer ranges (the empty stretches
// of a row beside the walls) are written by the whole wavefront, 64 cells per
// store.
constexpr uint32_t kOwnCells = 4;
constexpr uint32_t kTailBlocks = 64;

__global__ __launch_bounds__(kBlock) void k_cell_lb(uint32_t n, uint32_t n_cells,
                                                    const uint32_t* __restrict__ skeys,
                                                    uint32_t* __restrict__ lb, uint32_t key_blocks) {
  if (blockIdx.x >= key_blocks) {
    const uint32_t first = n == 0 ? 0u : skeys[n - 1] + 1u;
    const uint32_t stride = (gridDim.x - key_blocks) * kBlock;
    for (uint32_t c = first + (blockIdx.x - key_blocks) * kBlock + threadIdx.x; c <= n_cells; c += stride) lb[c] = n;
    return;
  }
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  uint32_t lo = 0, hi = 0;
  if (k < n) {
    lo = k == 0 ? 0u : skeys[k - 1] + 1u;
    hi = skeys[k] + 1u;
  }
  const uint32_t len = hi > lo ? hi - lo : 0u;
  if (len <= kOwnCells)
    for (uint32_t c = lo; c < hi; ++c) lb[c] = k;
  // wave-uniform loop over the lanes with long ranges
  uint64_t m = __ballot(len > kOwnCells);
  const uint32_t lane = __lane_id();
  while (m) {
    const int l = __builtin_ctzll(m);
    m &= m - 1;
    const uint32_t a = (uint32_t)__builtin_amdgcn_readlane((int)lo, l);
    const uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)hi, l);
    const uint32_t v = (uint32_t)__builtin_amdgcn_readlane((int)k, l);
    for (uint32_t c = a + lane; c < e; c += 64u) lb[c] = v;
  }
}

static void launch_cell_lb(Ctx& c, const uint32_t* skeys) {
  const uint32_t n = (uint32_t)c.n;
  const uint32_t key_blocks = (uint32_t)blocks_for(n);
  k_cell_lb<<<key_blocks + kTailBlocks, kBlock, 0, c.stream>>>(n, c.grid.n_cells, skeys, c.lb.as<uint32_t>(),
                                                               key_blocks);
  PR_HIP(hipGetLastError());
}

void neighbors_build(Ctx& c) {
  const uint32_t n = (uint32_t)c.n;
  if (!c.keys_valid) keys_from_positions(c);
  if (n == 0) {
    launch_cell_lb(c, nullptr);
    c.sorted = true; c.built = true;
    return;
  }
  // incremental when the state is still in the previous build's slot order
  // with fresh keys (right after a step)
  const int src = c.cur, dst = c.cur ^ 1;
  if (c.inc_ready && c.inc_fits() && !c.sort_radix) {
    incremental_sort(c);
  } else {
    if (c.inc_counts) {   // counts of a step this build does not continue
      PR_HIP(hipMemsetAsync(c.inc_cin(0), 0, c.inc_count_bytes(), c.stream));
      c.inc_counts = false;
    }
    if (c.sort_radix || !count_sort_fits(n, c.grid.n_cells) || !context_count_sort(c)) {
      radix_sort(c);
      const uint32_t* skeys = c.keys[c.cur_key].as<uint32_t>();
      const uint32_t* perm = c.vals[c.perm_buf].as<uint32_t>();
      {
        LaunchScope ls(&c, "reorder", reorder_bytes(c) * n);
        with_reorder_form(c, src, dst, [&](auto form, auto io) {
          using F = decltype(form);
          k_reorder<typename F::T, F::omega, F::probe, F::mixed><<<blocks_for(n), kBlock, 0, c.stream>>>(n, perm, skeys, io);
        });
        PR_HIP(hipGetLastError());
      }
      LaunchScope ls(&c, "cell_lb", 8.0 * n + 4.0 * c.grid.n_cells);
      launch_cell_lb(c, skeys);
    }
  }
  c.inc_ready = false;
  c.cur = dst;
  c.cur_ids ^= 1;
  c.sorted = true;
  c.built = true;
}

// ---------------------------------------------------------------------------
// id-order transfer helpers
// ---------------------------------------------------------------------------
// src_kind / dst_kind: 0 = double, 1 = float; comp and stride select one
// component of a packed element (stride 4 for double4/float4).

template <class T>
__global__ void k_scatter_ids(uint32_t n, const T* __restrict__ src, int stride, int comp,
                              const uint32_t* __restrict__ ids, double* __restrict__ out) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) out[ids[k]] = (double)src[(size_t)k * stride + comp];
}

// (of an upload: nothing when *bad is set, the field's values failed their check)
template <class T>
__global__ void k_gather_ids(uint32_t n, const double* __restrict__ in,
                             const uint32_t* __restrict__ ids, T* __restrict__ dst, int stride,
                             int comp, const uint32_t* __restrict__ bad) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n && *bad == 0u) dst[(size_t)k * stride + comp] = (T)in[ids[k]];
}

__global__ void k_scatter_keys(uint32_t n, const uint32_t* __restrict__ keys,
                               const uint32_t* __restrict__ ids, double* __restrict__ out) {
  uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k < n) out[ids[k]] = (double)keys[k];
}

void scatter_to_ids(Ctx& c, const void* src, int src_kind, int comp, double* d_out) {
  const uint32_t n = (uint32_t)c.n;
  if (!n) return;
  const uint32_t* ids = c.ids[c.cur_ids].as<uint32_t>();
  int stride = comp >= 0 ? (comp >= 100 ? 2 : 4) : 1;
  int cc = comp >= 100 ? comp - 100 : (comp >= 0 ? comp : 0);
  if (src_kind == 2) {
    k_scatter_keys<<<blocks_for(n), kBlock, 0, c.stream>>>(n, (const uint32_t*)src, ids, d_out);
  } else if (src_kind == 0) {
    k_scatter_ids<double><<<blocks_for(n), kBlock, 0, c.stream>>>(n, (const double*)src, stride, cc, ids, d_out);
  } else {
    k_scatter_ids<float><<<blocks_for(n), kBlock, 0, c.stream>>>(n, (const float*)src, stride, cc, ids, d_out);
  }
  PR_HIP(hipGetLastError());
}

void gather_from_ids(Ctx& c, const double* d_in, void* dst, int dst_kind, int comp) {
  const uint32_t n = (uint32_t)c.n;
  if (!n) return;
  const uint32_t* ids = c.ids[c.cur_ids].as<uint32_t>();
  const uint32_t* bad = c.flags.as<uint32_t>() + FLAG_COUNT;
  int stride = comp >= 0 ? (comp >= 100 ? 2 : 4) : 1;
  int cc = comp >= 100 ? comp - 100 : (comp >= 0 ? comp : 0);
  if (dst_kind == 0)
    k_gather_ids<double><<<blocks_for(n), kBlock, 0, c.stream>>>(n, d_in, ids, (double*)dst, stride, cc, bad);
  else
    k_gather_ids<float><<<blocks_for(n), kBlock, 0, c.stream>>>(n, d_in, ids, (float*)dst, stride, cc, bad);
  PR_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// eq1: force[i] += mass[j] (prestige/src/lib.rs:10) inside the loop of
// prestige/src/codegen/simple_cpu.rs:7-19.
// ---------------------------------------------------------------------------

// All pairs: thread t is particle id t, j runs over ids 0..n-1 in id order,
// exactly the generated loop.  force and mass are held in id order.
// Each force is one chain of dependent FP64 adds (8 cycles each), so the
// masses must reach every lane without costing issue slots or LDS bandwidth:
// each row of 16 lanes holds 16 consecutive masses, one per lane, and adds the
// k-th to all its lanes with a row broadcast in the instruction itself
// (acc = mass * 1 + acc, the same rounding as the add).  128 masses are held
// and the next 128 load meanwhile.  Read through LDS (16 bytes to 64 lanes is
// 8 cycles of a CU's LDS) the four wavefronts of a block took 13.4 cycles a
// mass at 10,000 particles, 57 us; this takes 8 cycles
// a mass, 35 us (60,000: 322 -> 199 us).
__device__ inline double add_row16(double acc, double x, double one) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %1, %2 row_newbcast:15 row_mask:0xf bank_mask:0xf"
      : "+v"(acc)
      : "v"(x), "v"(one));
  return acc;
}

constexpr uint32_t kPairBatch = 8;   // rows of 16 masses held
__global__ __launch_bounds__(64) void k_eq1_allpairs(uint32_t n, const double* __restrict__ mass,
                                                     double* __restrict__ force) {
  const uint32_t i = blockIdx.x * 64u + threadIdx.x, l = threadIdx.x & 15u;
  double acc = i < n ? force[i] : 0.0;   // every lane stays active: the broadcasts read them all
  const double one = 1.0;
  constexpr uint32_t kStep = 16u * kPairBatch;
  const uint32_t whole = n / kStep * kStep;
  double cur[kPairBatch], nxt[kPairBatch];
#pragma unroll
  for (uint32_t u = 0; u < kPairBatch; ++u) cur[u] = mass[min(16u * u + l, n - 1u)];
  for (uint32_t j0 = 0; j0 < whole; j0 += kStep) {
#pragma unroll
    for (uint32_t u = 0; u < kPairBatch; ++u) nxt[u] = mass[min(j0 + kStep + 16u * u + l, n - 1u)];
#pragma unroll
    for (uint32_t u = 0; u < kPairBatch; ++u) acc = add_row16(acc, cur[u], one);
#pragma unroll
    for (uint32_t u = 0; u < kPairBatch; ++u) cur[u] = nxt[u];
  }
  // the last n % 128 masses: whole rows from the registers, then one by one
  uint32_t j = whole;
#pragma unroll
  for (uint32_t u = 0; u < kPairBatch; ++u)
    if (j + 16u <= n) {
      acc = add_row16(acc, cur[u], one);
      j += 16u;
    }
  for (; j < n; ++j) acc += mass[j];
  if (i < n) force[i] = acc;
}

// Cells: j over the nine row runs of slot i, kept when |x_i - x_j|^2 < cutoff^2.
// force / mass are in id order; slot i updates force[ids[i]] only.
//
// One wavefront per block (64 consecutive slots).  Per row run the wavefront
// copies the union of its lanes' candidate ranges into LDS as FP32 offsets
// from its first slot in units of the cutoff (|q|^2 in .w), with their masses.
// Each lane then takes its own candidates in slot order with the dot form
// q.w - 2 s.q, which decides almost every pair: below 1 - m it lies inside the
// cutoff, at 1 + m or above outside, with m twice the rounding bound of the
// form (32 u (M^2 + M + 1), u = 2^-24, M the largest offset); a mass inside is
// added at once.  A wavefront in which some lane's candidate falls between (a
// few pairs in 10^5) takes the exact FP64 test for it.  So the pairs and the
// order are the plain loop's, and each force is its sum bit for bit.
// A union wider than the stage takes the exact test throughout, as do offsets too
// large for FP32.
// The masses come in slot order (smass[mstride j]): gathered by id in here they
// were 18 of a wavefront's loads of 64 scattered lines each, and what bounded it
// (236 us below).  Four candidates share the question whether any lane is in doubt.
// 1M random particles at 2.4 spacings: 191 us (masses in order 12 more);
// scanning into masks, walking the set bits and testing each exactly took 403
// (1.8M of a jittered dam break: 522 -> 344 with the masses).  What bounds it are
// the LDS reads, 24 bytes a candidate and lane, and instruction issue, five a
// candidate.  Where many pairs lie at the cutoff to seven digits (an undisturbed
// lattice with a lattice distance for a cutoff) the exact tests cost what the
// direct sums save: 395 -> 403.
constexpr uint32_t kEq1Stage = 256;
constexpr uint32_t kEq1Batch = 4;   // candidates in flight (the exact path picks among four)

template <class T4>
__global__ __launch_bounds__(64) void k_eq1_cells(uint32_t n, const T4* __restrict__ pos,
                                                  const uint32_t* __restrict__ ids,
                                                  const uint32_t* __restrict__ skeys,
                                                  const uint32_t* __restrict__ lb, Grid g, double c2,
                                                  double inv_cut, const double* __restrict__ smass, uint32_t mstride,
                                                  double* __restrict__ force, uint32_t n_tiles) {
#pragma clang fp contract(off)
  __shared__ float4 s_q[kEq1Stage + kEq1Batch];   // (a batch may read past the stage's end)
  __shared__ double s_m[kEq1Stage + kEq1Batch];
  const uint32_t tile = xcd_tile(blockIdx.x);
  if (tile >= n_tiles) return;
  const uint32_t lane = threadIdx.x, wbase = tile * 64u, i = wbase + lane;
  const bool live = i < n;
  const uint32_t self = live ? i : wbase;
  const T4 pi = pos[self];
  const T4 p0 = pos[wbase];
  const double xr = (double)p0.x, yr = (double)p0.y, zr = (double)p0.z;
  auto offset = [&](const T4& p) {
    float4 q = make_float4((float)(((double)p.x - xr) * inv_cut), (float)(((double)p.y - yr) * inv_cut),
                           (float)(((double)p.z - zr) * inv_cut), 0.0f);
    q.w = __builtin_fmaf(q.x, q.x, __builtin_fmaf(q.y, q.y, q.z * q.z));
    return q;
  };
  auto exact = [&](uint32_t j) {
    const T4 pj = pos[j];
    const double ex = (double)pi.x - (double)pj.x, ey = (double)pi.y - (double)pj.y, ez = (double)pi.z - (double)pj.z;
    return ex * ex + ey * ey + ez * ez < c2;
  };
  const uint32_t me = ids[self];
  double acc = live ? force[me] : 0.0;
  const uint32_t nx = (uint32_t)g.dims[0], ny = (uint32_t)g.dims[1], nz = (uint32_t)g.dims[2];
  const uint32_t key = skeys[self];
  const int cx = (int)(key % nx), cy = (int)((key / nx) % ny), cz = (int)(key / (nx * ny));
  const int x0 = cx > 0 ? cx - 1 : 0, x1 = cx < (int)nx - 1 ? cx + 1 : (int)nx - 1;
  // the nine row runs' ranges, read at once
  uint32_t j0[9], len[9];
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    const int zz = cz + r / 3 - 1, yy = cy + r % 3 - 1;
    const bool ok = live && zz >= 0 && zz < (int)nz && yy >= 0 && yy < (int)ny;
    const uint32_t row = ok ? ((uint32_t)zz * ny + (uint32_t)yy) * nx : 0u;
    j0[r] = lb[row + (uint32_t)x0];
    len[r] = ok ? lb[row + (uint32_t)x1 + 1u] - j0[r] : 0u;
  }
  const float4 so = offset(pi);
  const float ax = -2.0f * so.x, ay = -2.0f * so.y, az = -2.0f * so.z;
  const float ss_max = wave_max_pos(live ? so.w : 0.0f);
#pragma unroll
  for (int r = 0; r < 9; ++r) {
    // union of the lanes' ranges: slots are in key order, so the first and
    // last lane with candidates bound it
    const uint64_t any = __ballot(len[r] != 0u);
    if (any == 0ull) continue;
    const uint32_t base = (uint32_t)__builtin_amdgcn_readlane((int)j0[r], __builtin_ctzll(any));
    const uint32_t span = (uint32_t)__builtin_amdgcn_readlane((int)(j0[r] + len[r]), 63 - __builtin_clzll(any)) - base;
    if (span > kEq1Stage) {
      for (uint32_t b = 0; b < len[r]; ++b)
        if (exact(j0[r] + b)) acc += smass[(size_t)mstride * (j0[r] + b)];
      continue;
    }
    float mq = 0.0f;
    for (uint32_t kk = lane; kk < span; kk += 64u) {
      const float4 q = offset(pos[base + kk]);
      s_q[kk] = q;
      s_m[kk] = smass[(size_t)mstride * (base + kk)];
      mq = q.w > mq ? q.w : mq;
    }
    const float m2 = fmaxf(ss_max, wave_max_pos(mq));
    const float margin = 0x1.0p-18f * (m2 + __builtin_sqrtf(m2) + 1.0f);
    // offsets of more than 2^50 cutoffs could overflow in the form: then no pair is
    // decided here (every comparison with a NaN is false)
    const bool far = !(m2 < 0x1.0p100f);
    const float lo = far ? __builtin_nanf("") : (1.0f - margin) - so.w;
    const float hi = far ? __builtin_nanf("") : (1.0f + margin) - so.w;
    __builtin_amdgcn_wave_barrier();   // one wavefront: its LDS operations complete in order
    const uint32_t first = j0[r] - base;
    auto batch = [&](uint32_t b, uint32_t cnt) {
      float v[kEq1Batch];
      double m[kEq1Batch];
#pragma unroll
      for (uint32_t u = 0; u < kEq1Batch; ++u) {
        const float4 q = s_q[first + b + u];
        v[u] = __builtin_fmaf(ax, q.x, __builtin_fmaf(ay, q.y, __builtin_fmaf(az, q.z, q.w)));
        if (u >= cnt) v[u] = 0x1.0p127f;   // past the run: outside
        m[u] = s_m[first + b + u];
      }
      uint64_t open = 0;   // lanes that cannot tell
#pragma unroll
      for (uint32_t u = 0; u < kEq1Batch; ++u) open |= __ballot(v[u] < lo) ^ __ballot(!(v[u] >= hi));
      if (open == 0ull) {
#pragma unroll
        for (uint32_t u = 0; u < kEq1Batch; ++u)
          if (v[u] < lo) {
            acc += m[u];
            asm volatile("" : "+v"(acc));   // an add under the lane mask; as a select it costs two moves more
          }
      } else {
#pragma unroll 1
        for (uint32_t u = 0; u < kEq1Batch; ++u) {
          const float w = u == 0u ? v[0] : (u == 1u ? v[1] : (u == 2u ? v[2] : v[3]));
          const double mu = u == 0u ? m[0] : (u == 1u ? m[1] : (u == 2u ? m[2] : m[3]));
          if (u < cnt && (w < lo || (!(w >= hi) && exact(j0[r] + b + u)))) acc += mu;
        }
      }
    };
    uint32_t b = 0;
    for (; b + kEq1Batch <= len[r]; b += kEq1Batch) batch(b, kEq1Batch);
    if (b < len[r]) batch(b, len[r] - b);
    __builtin_amdgcn_wave_barrier();
  }
  if (live) force[me] = acc;
}

__global__ __launch_bounds__(kBlock) void k_eq1_masses(uint32_t n, const uint32_t* __restrict__ ids,
                                                       const double* __restrict__ mass, double* __restrict__ smass) {
  const uint32_t k = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (k < n) smass[k] = mass[ids[k]];
}

void eq1_eval(Ctx& c, int loop, double cutoff) {
  const uint32_t n = (uint32_t)c.n;
  PR_CHECK(c.have_force && c.have_mass, PRESTIGE_E_STATE, "eq1 needs fields 'force' and 'mass' uploaded");
  if (!n) return;
  if (loop == PRESTIGE_LOOP_ALLPAIRS) {
    LaunchScope ls(&c, "eq1_allpairs", 24.0 * n);
    k_eq1_allpairs<<<blocks_for(n, 64), 64, 0, c.stream>>>(n, c.mass.as<double>(), c.force.as<double>());
    PR_HIP(hipGetLastError());
    return;
  }
  PR_CHECK(loop == PRESTIGE_LOOP_CELLS, PRESTIGE_E_INVALID, "unknown loop mode");
  PR_CHECK(cutoff > 0.0 && cutoff <= c.grid.cs, PRESTIGE_E_INVALID, "cutoff must be in (0, cell_size]");
  if (!c.sorted) neighbors_build(c);
  LaunchScope ls(&c, "eq1_cells", 56.0 * n);
  const uint32_t* ids = c.ids[c.cur_ids].as<uint32_t>();
  const uint32_t tiles = blocks_for(n, 64);
  double* smass = c.scratch.as<double>();
  k_eq1_masses<<<blocks_for(n), kBlock, 0, c.stream>>>(n, ids, c.mass.as<double>(), smass);
  PR_HIP(hipGetLastError());
  if (c.desc.precision == PRESTIGE_F32)
    k_eq1_cells<float4><<<tile_grid(tiles), 64, 0, c.stream>>>(
        n, c.pos[c.cur].as<float4>(), ids, c.keys[c.cur_key].as<uint32_t>(), c.lb.as<uint32_t>(),
        c.grid, cutoff * cutoff, 1.0 / cutoff, smass, 1u, c.force.as<double>(), tiles);
  else
    k_eq1_cells<double4><<<tile_grid(tiles), 64, 0, c.stream>>>(
        n, c.pos[c.cur].as<double4>(), ids, c.keys[c.cur_key].as<uint32_t>(), c.lb.as<uint32_t>(),
        c.grid, cutoff * cutoff, 1.0 / cutoff, smass, 1u, c.force.as<double>(), tiles);
  PR_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// eq1 over the cell iterator without allocating (prestige_eq1_cells_noalloc)
// ---------------------------------------------------------------------------
// The same kernels as prestige_eval_equation(PRESTIGE_EQ1, PRESTIGE_LOOP_CELLS)
// on a fresh context (cell keys, counting sort with the positions moved, the
// eq1 gather), on the caller's device arrays, with every
// intermediate array in one file-scope device array: `scratch`.  It holds
// keys, sorted keys, permutation and arrival numbers (16 B per particle), the
// positions in order of arrival and sorted (64 B), the cell table (4 B per cell + 4), its tile totals
// and the error flags, each at a 256-byte boundary, sized for at
// most kNoAllocMaxN particles and kNoAllocMaxCells cells.  Each device holds
// its own copy; host code reaches it only through the address
// hipGetSymbolAddress gives on that device (noalloc_scratch), never through
// the array's name.  Every call on a device reuses that device's copy, so
// calls that overlap on one device race; each call clears what must start
// at zero (the flags) with a kernel.
constexpr uint64_t kNoAllocMaxN = 1ull << 20;
constexpr uint64_t kNoAllocMaxCells = 1ull << 22;

constexpr uint64_t na_round(uint64_t b) { return (b + 255ull) & ~255ull; }
constexpr uint64_t kNaKeys = 0;                                               // keys, sorted keys: 2 x 4 N
constexpr uint64_t kNaVals = kNaKeys + 2 * na_round(4 * kNoAllocMaxN);        // permutation, arrivals: 2 x 4 N
constexpr uint64_t kNaPos = kNaVals + 2 * na_round(4 * kNoAllocMaxN);         // double4 x N, twice
constexpr uint64_t kNaLb = kNaPos + 2 * na_round(32 * kNoAllocMaxN);          // cells + 1
constexpr uint64_t kNaTot = kNaLb + na_round(4 * (kNoAllocMaxCells + 1));     // a total per tile of cells
constexpr uint64_t kNaFlags = kNaTot + na_round(4ull * (kNoAllocMaxCells / kCellTile + 1));
constexpr uint64_t kNoAllocBytes = kNaFlags + na_round(4ull * FLAG_COUNT);

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

__global__ __launch_bounds__(kBlock) void k_count_soa(uint32_t n, const double* __restrict__ x,
                                                      const double* __restrict__ y, const double* __restrict__ z,
                                                      Grid g, uint32_t* __restrict__ keys, uint32_t* __restrict__ cnt,
                                                      uint32_t* __restrict__ arr, uint32_t* flags) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  const bool live = i < n;
  const uint32_t key = live ? cell_key_of(x[i], y[i], z[i], g, flags) : 0u;
  const uint32_t a = cell_arrival(cnt, key, live, nullptr);
  if (live) {
    keys[i] = key;
    arr[i] = a;
  }
}

// The points in order of arrival, with (slot, key) in .w: one write of 32 bytes
// to a scattered place each, where reading them from there in cell order takes
// three (1M points in no order: 19 us and 18 for k_count_rank_soa; lists and
// k_count_place 15 and 65).
__global__ __launch_bounds__(kBlock) void k_count_scatter_soa(uint32_t n, const double* __restrict__ x,
                                                              const double* __restrict__ y,
                                                              const double* __restrict__ z,
                                                              const uint32_t* __restrict__ keys,
                                                              const uint32_t* __restrict__ arr,
                                                              const uint32_t* __restrict__ lb,
                                                              double4* __restrict__ upos) {
  const uint32_t i = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (i >= n) return;
  const uint32_t key = keys[i];
  upos[lb[key] + arr[i]] = make_double4(x[i], y[i], z[i], __longlong_as_double((long long)((uint64_t)key << 32 | i)));
}

// Then by slot within each cell (k_count_place for points that are in cell order
// already: what it reads and writes lies close together; the ids of a first
// build are the permutation itself).
__global__ __launch_bounds__(kBlock) void k_count_rank_soa(uint32_t n, const double4* __restrict__ upos,
                                                           const uint32_t* __restrict__ lb,
                                                           const double* __restrict__ mass,
                                                           double4* __restrict__ spos, uint32_t* __restrict__ skeys,
                                                           uint32_t* __restrict__ perm) {
  const uint32_t k = blockIdx.x * (uint32_t)kBlock + threadIdx.x;
  if (k >= n) return;
  const double4 p = upos[k];
  const uint64_t w = (uint64_t)__double_as_longlong(p.w);
  const uint32_t key = (uint32_t)(w >> 32), i = (uint32_t)w;
  const uint32_t* slot = reinterpret_cast<const uint32_t*>(upos) + 6;   // entry q's slot is slot[8 q]
  const uint32_t end = lb[key + 1u];
  uint32_t q = lb[key], pos = q;
  for (; q + 4u <= end; q += 4u) {
    uint32_t v[4];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) v[k] = slot[8u * (size_t)(q + k)];
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) pos += v[k] < i ? 1u : 0u;
  }
  for (; q < end; ++q) pos += slot[8u * (size_t)q] < i ? 1u : 0u;
  spos[pos] = make_double4(p.x, p.y, p.z, mass[i]);
  skeys[pos] = key;
  perm[pos] = i;
}

// Device address of this device's scratch, looked up once per device with
// that device current.
static void* noalloc_scratch(int device) {
  static std::mutex mu;
  static void* addr[64] = {};
  PR_CHECK(device >= 0 && device < 64, PRESTIGE_E_INVALID, "device index out of range");
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    void* p = nullptr;
    PR_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    PR_CHECK(p != nullptr, PRESTIGE_E_HIP, "hipGetSymbolAddress returned no address for the scratch array");
    addr[device] = p;
  }
  return addr[device];
}

static void eq1_cells_noalloc(const double* x, const double* y, const double* z, const double* mass, double* force,
                              uint64_t n64, const double lo[3], const double hi[3], double cell_size, double cutoff,
                              hipStream_t st) {
  PR_CHECK(lo != nullptr && hi != nullptr, PRESTIGE_E_INVALID, "null grid bounds");
  const Grid g = make_grid(lo, hi, cell_size);
  PR_CHECK(cutoff > 0.0 && cutoff <= g.cs, PRESTIGE_E_INVALID, "cutoff must be in (0, cell_size]");
  PR_CHECK(n64 <= kNoAllocMaxN, PRESTIGE_E_CAPACITY,
           "n = " + std::to_string(n64) + " exceeds the " + std::to_string(kNoAllocMaxN) +
               " particles the allocation-free scratch holds");
  PR_CHECK(g.n_cells <= kNoAllocMaxCells, PRESTIGE_E_CAPACITY,
           "the grid has " + std::to_string(g.n_cells) + " cells, more than the " + std::to_string(kNoAllocMaxCells) +
               " the allocation-free scratch holds");
  if (n64 == 0) return;
  PR_CHECK(x && y && z && mass && force, PRESTIGE_E_INVALID, "null particle array");
  const uint32_t n = (uint32_t)n64;
  int dev = 0;
  PR_HIP(hipGetDevice(&dev));
  unsigned char* base = static_cast<unsigned char*>(noalloc_scratch(dev));
  uint32_t* flags = reinterpret_cast<uint32_t*>(base + kNaFlags);
  uint32_t* keys = reinterpret_cast<uint32_t*>(base + kNaKeys);
  uint32_t* skeys = reinterpret_cast<uint32_t*>(base + kNaKeys + na_round(4 * kNoAllocMaxN));
  uint32_t* perm = reinterpret_cast<uint32_t*>(base + kNaVals);
  uint32_t* arr = reinterpret_cast<uint32_t*>(base + kNaVals + na_round(4 * kNoAllocMaxN));
  double4* upos = reinterpret_cast<double4*>(base + kNaPos);
  double4* spos = reinterpret_cast<double4*>(base + kNaPos + na_round(32 * kNoAllocMaxN));
  uint32_t* lb = reinterpret_cast<uint32_t*>(base + kNaLb);
  uint32_t* tot = reinterpret_cast<uint32_t*>(base + kNaTot);
  k_count_clear<<<blocks_for(g.n_cells + 1u), kBlock, 0, st>>>(g.n_cells + 1u, lb, FLAG_COUNT, flags);
  PR_HIP(hipGetLastError());
  k_count_soa<<<blocks_for(n), kBlock, 0, st>>>(n, x, y, z, g, keys, lb, arr, flags);
  PR_HIP(hipGetLastError());
  count_table(nullptr, g.n_cells, lb, tot, Crowd{}, st);
  k_count_scatter_soa<<<blocks_for(n), kBlock, 0, st>>>(n, x, y, z, keys, arr, lb, upos);
  PR_HIP(hipGetLastError());
  k_count_rank_soa<<<blocks_for(n), kBlock, 0, st>>>(n, upos, lb, mass, spos, skeys, perm);
  PR_HIP(hipGetLastError());
  const uint32_t tiles = blocks_for(n, 64);
  k_eq1_cells<double4><<<tile_grid(tiles), 64, 0, st>>>(n, spos, perm, skeys, lb, g, cutoff * cutoff, 1.0 / cutoff,
                                                        &spos->w, 4u, force, tiles);
  PR_HIP(hipGetLastError());
  uint32_t h[FLAG_COUNT] = {0, 0, 0, 0};
  PR_HIP(hipMemcpyAsync(h, flags, sizeof(h), hipMemcpyDeviceToHost, st));
  PR_HIP(hipStreamSynchronize(st));
  PR_CHECK(h[FLAG_DOMAIN] == 0u, PRESTIGE_E_DOMAIN, "a particle lies outside the cell grid");
}

}  // namespace prestige

extern "C" prestige_status prestige_eq1_cells_noalloc(const double* x, const double* y, const double* z,
                                                      const double* mass, double* force, uint64_t n,
                                                      const double grid_lo[3], const double grid_hi[3],
                                                      double cell_size, double cutoff, void* stream) {
  try {
    prestige::eq1_cells_noalloc(x, y, z, mass, force, n, grid_lo, grid_hi, cell_size, cutoff,
                                static_cast<hipStream_t>(stream));
    prestige::set_context_free_error("");
    return PRESTIGE_OK;
  } catch (const prestige::Error& e) {
    prestige::set_context_free_error(e.what());
    return e.code;
  } catch (const std::exception& e) {
    prestige::set_context_free_error(e.what());
    return PRESTIGE_E_INVALID;
  } catch (...) {
    prestige::set_context_free_error("unknown C++ exception");
    return PRESTIGE_E_INVALID;
  }
}
