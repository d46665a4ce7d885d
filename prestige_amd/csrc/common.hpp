// common.hpp — internal types of libprestige_hip.so (not part of the C ABI).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <map>
#include <memory>
#include <cstring>
#include <stdexcept>
#include <string>
#include <type_traits>
#include <utility>
#include <vector>

#include "../../include/prestige_hip.h"

namespace prestige {

// Error carrying a prestige_status across internal C++ code; converted to a
// status code at the C ABI.
struct Error : std::runtime_error {
  prestige_status code;
  Error(prestige_status c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define PR_HIP(call)                                                                 \
  do {                                                                               \
    hipError_t e_ = (call);                                                          \
    if (e_ != hipSuccess)                                                            \
      throw ::prestige::Error(e_ == hipErrorOutOfMemory ? PRESTIGE_E_OOM : PRESTIGE_E_HIP, \
                              std::string(#call) + ": " + hipGetErrorString(e_));    \
  } while (0)

#define PR_CHECK(cond, code, msg)                                   \
  do {                                                              \
    if (!(cond)) throw ::prestige::Error((code), (msg));            \
  } while (0)

// Device flags written by kernels on error paths only.
// FLAG_CFL: a moving particle outran the step (WCSPH: dt (c0 + |v|) > h / 2;
// DEM: dt |v| > r / 4).
enum FlagSlot : int { FLAG_DOMAIN = 0, FLAG_CAPACITY = 1, FLAG_NONFINITE = 2, FLAG_CFL = 3, FLAG_COUNT = 4 };

// Cell grid: key = (cz*ny + cy)*nx + cx, c = floor((x - lo) * inv_cs).
struct Grid {
  double lo[3];
  double cs;
  double inv_cs;
  double off_scale;   // MIXED offsets are (x - origin) * off_scale (1/h for WCSPH, 1 for DEM)
  int32_t dims[3];
  uint32_t n_cells;
};

// Grid of the box [lo, hi) in cells of size cs: dims = ceil((hi - lo) / cs)
// per axis (every context and the allocation-free entry point build it
// here, so their keys agree bit for bit).
inline Grid make_grid(const double lo[3], const double hi[3], double cs) {
  Grid g{};
  PR_CHECK(cs > 0.0 && cs < 1.0e300, PRESTIGE_E_INVALID, "cell_size must be finite and > 0");
  for (int a = 0; a < 3; ++a) {
    g.lo[a] = lo[a];
    const double span = hi[a] - lo[a];
    PR_CHECK(span > 0.0, PRESTIGE_E_INVALID, "grid_hi must exceed grid_lo on every axis");
    const double cells = __builtin_ceil(span / cs);
    PR_CHECK(cells >= 1.0 && cells < 2.0e9, PRESTIGE_E_INVALID, "grid has too many cells along an axis");
    g.dims[a] = (int32_t)cells;
  }
  g.cs = cs;
  g.inv_cs = 1.0 / cs;
  const double nc = (double)g.dims[0] * (double)g.dims[1] * (double)g.dims[2];
  PR_CHECK(nc < 4.0e9, PRESTIGE_E_INVALID, "grid has more than 4e9 cells");
  g.n_cells = (uint32_t)nc;
  g.off_scale = 1.0;
  return g;
}

// Constants of the WCSPH bodies, derived once on the host from the
// descriptor.  Every device form reads the same FP64 values (FP32 forms
// round them once).
struct SphConst {
  double h, inv_h, H2, eps2, inv_rho0, B, alpha_c0, msig, msh, dt;
  double g[3];
  double cfl_v2;   // largest |v|^2 with dt (c0 + |v|) <= h / 2 (negative: dt alone breaks it)
};

struct DemConst {
  double kn, kt, mu, two_zeta, neg_inv_kt, dt;
  double g[3];
  double wall_lo[3], wall_hi[3];
  uint32_t wall_mask;
  uint32_t max_contacts;
};

// Owned device allocation.
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    bytes = 0;
  }
  void alloc(size_t b) {
    if (b == bytes && p) return;
    release();
    if (b == 0) return;
    hipError_t e = hipMalloc(&p, b);
    if (e != hipSuccess) {
      p = nullptr;
      throw Error(PRESTIGE_E_OOM, "hipMalloc(" + std::to_string(b) + " bytes) failed: " + hipGetErrorString(e));
    }
    bytes = b;
  }
  template <class T> T* as() const { return static_cast<T*>(p); }
};

// Per-kernel HIP-event timing on the context stream.
struct KernelStat {
  const char* name;
  double total_ms = 0.0;
  uint64_t launches = 0;
  double bytes_per_launch = 0.0;
};

struct Timing {
  bool enabled = false;
  std::vector<KernelStat> stats;
  struct Pending { hipEvent_t a, b; size_t stat; };
  std::vector<Pending> pending;
  std::vector<hipEvent_t> pool;
  hipEvent_t get_event();
  size_t stat_index(const char* name, double bytes);
  void flush();   // collect elapsed times of completed pairs (synchronises on each)
  void clear();
  ~Timing();
};

struct Ctx;
// Whether a context of n slots builds in one launch after a step (neighbors.hip).
bool inc_in_one(uint64_t n, size_t cell_tiles);

// What the step kernels leave for the next build's incremental sort.  A slot
// whose particle changes cell ("moved", fixed particles never do) counts into
// its new cell (cin) and out of its old one (cout), into the same totals per
// tile of kCellTile cells (tin, tout), and is linked into its new cell's list:
// head[c] holds (epoch << 32 | last slot linked), next[slot] the slot linked
// before it (kListEnd for the first of this epoch, so heads need no clearing but
// when the 32-bit epochs start again, at 1).  Word w of mask has bit l set when
// slot 64 w + l moved.  What came less what left is also taken per 2^net_shift
// cells (net): per kCellGroup where the build is one launch, else per kTileGroup
// tiles.
constexpr uint32_t kCellTile = 1024;
constexpr uint32_t kCellGroup = 32;    // 2^5
constexpr uint32_t kTileGroup = 256;   // 2^8 tiles of 2^10 cells
constexpr uint32_t kListEnd = 0xFFFFFFFFu;
// Runaways (particles that outran the time step, which is an error) one cell's
// list takes in one step; the others stay in their old cells.  A build walks a
// cell's list once for every slot of the cell, a dependent load (some 0.4 us) an
// entry: 65,536 take 30 ms.  Particles within the step's bound are all listed: they
// enter in such numbers only where as many share the cell, and the contact pass
// tests each of those against all others (more than 128 in a row of cells end a
// WCSPH step).
constexpr uint32_t kMaxIn = 1u << 16;
struct MovedOut {
  uint64_t* mask;
  uint32_t *cin, *cout, *tin, *tout, *net;
  uint64_t* head;
  uint32_t* next;
  uint32_t epoch, net_shift;
};
// Slot i goes from cell old_key to cell key: record it; false when it stays
// (key is then old_key).
__device__ inline bool move_to_cell(const MovedOut& mo, uint32_t i, uint32_t old_key, uint32_t& key, bool runaway) {
  if (key == old_key) return false;
  if (!mo.cin) return true;   // a context without them sorts by the keys alone
  if (atomicAdd(&mo.cin[key], 1u) >= kMaxIn && runaway) {
    atomicSub(&mo.cin[key], 1u);
    key = old_key;
    return false;
  }
  atomicAdd(&mo.cout[old_key], 1u);
  atomicAdd(&mo.tin[key / kCellTile], 1u);
  atomicAdd(&mo.tout[old_key / kCellTile], 1u);
  if (key >> mo.net_shift != old_key >> mo.net_shift) {
    atomicAdd(&mo.net[key >> mo.net_shift], 1u);
    atomicSub(&mo.net[old_key >> mo.net_shift], 1u);
  }
  const unsigned long long mine = ((unsigned long long)mo.epoch << 32) | i;
  const unsigned long long last = atomicExch(reinterpret_cast<unsigned long long*>(&mo.head[key]), mine);
  mo.next[i] = (uint32_t)(last >> 32) == mo.epoch ? (uint32_t)last : kListEnd;
  return true;
}

// Hand a buffer a step just wrote to an adjoint record without copying: the
// next step only writes into the context side of the swap before reading it.
inline void take_buffer(DevBuf& ctx_buf, DevBuf& rec_buf) {
  if (rec_buf.bytes != ctx_buf.bytes) rec_buf.alloc(ctx_buf.bytes);
  std::swap(ctx_buf.p, rec_buf.p);
}

// Records `name` around one launch when timing is on.
struct LaunchScope {
  Ctx* ctx;
  size_t stat;
  hipEvent_t a = nullptr, b = nullptr;
  LaunchScope(Ctx* c, const char* name, double bytes);
  ~LaunchScope() noexcept(false);
};

// One device-to-device copy of a list (copy_many allocates dst).
struct Copy {
  DevBuf* dst;
  DevBuf* src;
  size_t bytes;
};

// Device copy of the full integration state (used as an adjoint checkpoint).
struct Snapshot {
  DevBuf pos, vel, omega, ids, keys;
  DevBuf hcnt, hid, hxi, wxi;   // DEM contact history
  int cur = 0, cur_ids = 0, cur_key = 0, cur_hist = 0;
  bool sorted = false, keys_valid = false, built = false;
};

// What the reverse sweep needs from one forward step: the sorted pre-step
// pair geometry, the gather outputs, and the frozen neighbour structure.
struct StepRecord {
  DevBuf gpos, gvel, gom, rp, ids, perm, nmeta, nword;
  DevBuf hcnt, hid, hxi, wxi;   // DEM history read by the step
  DevBuf hcnt_out, hid_out;     // DEM contacts the step found (its frozen contact lists)
  DevBuf state_pos, state_vel, state_om;   // DEM FP64 pre-step state (sorted)
};

// Adjoint tape: checkpoints every `every` steps of an nsteps forward run.
struct Tape {
  bool valid = false;
  bool last_recorded = false;   // rec holds the last segment of the taped forward
  uint32_t nsteps = 0, every = 0;
  std::vector<std::unique_ptr<Snapshot>> ckpt;   // state before step s * every
  size_t n_ckpt = 0;                             // checkpoints in use (ckpt keeps its buffers)
  std::unique_ptr<Snapshot> final_state;
  std::vector<std::unique_ptr<StepRecord>> rec;  // reused across segments
  DevBuf xb, vb, xb2, vb2, cvec, xbf, rhob, partial, acc, seeds, wb, wb2;
  DevBuf hb[2], wallb[2], slot_of;   // DEM history adjoints (ping-pong), id -> slot
  DevBuf wallm[2];              // walls a step touched, by particle id (bits 0-5)
  // Start a new tape; checkpoint buffers are kept and reused.
  void clear() {
    n_ckpt = 0;
    valid = false;
    last_recorded = false;
  }
  Snapshot& next_ckpt() {
    if (n_ckpt == ckpt.size()) ckpt.emplace_back(new Snapshot());
    return *ckpt[n_ckpt++];
  }
};

// Words of Ctx::note: what a field check found (kNoteField + bit), a first build's (Crowd).
enum Note : int { kNoteField = 0, kNoteCrowd = 3, kNotes = 4 };

struct Ctx {
  Ctx() = default;
  Ctx(const Ctx&) = delete;
  Ctx& operator=(const Ctx&) = delete;
  ~Ctx() {
    if (pin) (void)hipHostFree(pin);
    if (ring) (void)hipHostFree(ring);
    for (auto e : ring_ev) (void)hipEventDestroy(e);
  }
  prestige_desc desc{};
  int device = 0;
  hipStream_t stream = nullptr;
  uint64_t n = 0, n_moving = 0;
  Grid grid{};
  SphConst sph{};
  DemConst dem{};
  std::string err;

  // slot bookkeeping: cur = buffer (0/1) holding the newest positions and
  // velocities; `sorted` = cur is in key order of the last build;
  // `keys_valid` = keys[cur_key] hold the cell keys of buffer cur.
  int cur = 0;
  bool sorted = false;
  bool keys_valid = false;
  bool built = false;
  int cur_key = 0;

  // state, ping-pong pairs (element type depends on precision)
  DevBuf pos[2], vel[2];         // double4 (F64, MIXED) or float4 (F32); DEM: pos.w = radius, vel.w = mass
  DevBuf omega[2];               // DEM: double4 / float4
  DevBuf ids[2];                 // uint32 original id per slot
  int cur_ids = 0;
  DevBuf keys[2], vals[2];       // radix-sort ping-pong
  int perm_buf = 0;              // which vals[] holds the last permutation
  DevBuf sort_hist, sort_tot;    // per-tile digit counts, per-digit totals
  // incremental sort (MovedOut): moved-slot mask, links per slot, the spare
  // cell table, and in one buffer the list heads per cell and the counts cin,
  // cout (inc_tiles * kCellTile each), net (inc_nets), tin, tout (inc_tiles each).  Where the build is one launch there are two sets of
  // counts: a step writes set inc_set, its build reads it and clears the other.
  // A context they do not fit has the mask only, and every build sorts anew.
  DevBuf inc_mask, inc_next, lb_spare, inc_cells;
  size_t inc_tiles = 0;
  bool inc_fits() const { return inc_cells.p != nullptr; }
  uint64_t* inc_head() const { return inc_cells.as<uint64_t>(); }
  size_t inc_head_bytes() const { return inc_tiles * kCellTile * 8; }
  uint32_t inc_net_shift() const { return inc_one ? 5u : 18u; }
  size_t inc_nets() const { return ((inc_tiles * kCellTile - 1) >> inc_net_shift()) + 1; }
  size_t inc_set_words() const { return (inc_tiles * (2 * kCellTile + 2) + inc_nets() + 3) / 4 * 4; }
  uint32_t* inc_cin(int set) const {
    return reinterpret_cast<uint32_t*>(inc_cells.as<char>() + inc_head_bytes()) + set * inc_set_words();
  }
  uint32_t* inc_cout(int set) const { return inc_cin(set) + inc_tiles * kCellTile; }
  uint32_t* inc_net(int set) const { return inc_cout(set) + inc_tiles * kCellTile; }
  uint32_t* inc_tin(int set) const { return inc_net(set) + inc_nets(); }
  uint32_t* inc_tout(int set) const { return inc_tin(set) + inc_tiles; }
  size_t inc_count_bytes() const { return (inc_one ? 2 : 1) * inc_set_words() * 4; }   // from inc_cin(0) on
  bool inc_one = false;          // the build after a step is one launch
  int inc_set = 0;
  uint32_t inc_epoch = 0;        // of the last step (PRESTIGE_EPOCH starts it elsewhere, for tests)
  bool inc_ready = false;        // keys[cur_key] are the next keys of the last build's slots
  bool inc_counts = false;       // a step's counts are waiting (a build that does not use them clears them)
  bool sort_radix = false;       // PRESTIGE_SORT=radix: every build is a radix sort (comparisons and tests)
  DevBuf lb;                     // n_cells + 1
  // WCSPH wall particles far from the fluid (DryWalls): cell stamps (n_cells),
  // last dry pass per particle id, pass counter, the pass the stamps describe,
  // and whether steps must leave every particle usable masks (adjoint records)
  DevBuf movcell, dry_pass, rp_id, pres_id;
  uint32_t dens_pass = 16, stamp_pass = 0;
  bool record_all = false;
  bool dry_reuse = true;         // PRESTIGE_DRY=off turns the reuse off (comparisons and tests)
  void forget_dry() { dens_pass += 2; }   // state changed outside a step
  DevBuf flags;                  // FLAG_COUNT uint32, then the field check's word and a first build's (Crowd)
  void* pin = nullptr;                       // pinned block for small transfers
  size_t pin_bytes = 0;
  // pinned words that kernels leave for the host (host and device address)
  uint32_t *note = nullptr, *note_dev = nullptr;
  bool take_note(int k) {   // reads and clears; after the kernel has been waited for
    volatile uint32_t* w = note + k;
    const bool set = *w != 0u;
    if (set) *w = 0u;
    return set;
  }
  uint32_t count_builds = 0;                 // first builds that asked for a crowded cell (Crowd)
  void* ring = nullptr;                      // pinned chunks of large ones, from the first on
  std::vector<hipEvent_t> ring_ev;
  // gather outputs
  DevBuf rp;                     // (rho, p/rho^2) per slot: double2 or float2
  DevBuf pres;                   // p per slot (double or float)
  DevBuf rp64, pres64;           // MIXED with PRESTIGE_FLAG_DENSITY_F64: the FP64 density outputs
  // PRESTIGE_FLAG_DEM_EVENTS: per particle id, step-weighted sums of contact
  // and slip counts (2 n uint32); steps counted since the last position
  // upload; weight of the step being run (0: not recording)
  DevBuf events;
  uint32_t ev_steps = 0, ev_weight = 0;
  DevBuf acc;                    // a per slot (double4 / float4)
  // MIXED form gather copies
  DevBuf off32, vel32, om32;     // float4: offset from cell origin (cell x in .w); velocity
                                 // (mass in .w); DEM angular velocity (radius in .w)
  // row-run masks of the last density pass: run r of slot i has (first
  // candidate slot, candidate count) at nmeta[r n + i] (uint2) and its hit
  // words at nword[(4 r + w) n + i] (uint32, written for 32 w < count)
  DevBuf nmeta, nword;
  // WCSPH gathers with four lanes per particle (sph_quad.hpp) and their
  // neighbour lists and counts.  PRESTIGE_QUAD=on|off overrides the choice by
  // size (comparisons and tests).
  bool quad = false;
  DevBuf nlist, ncnt;
  // eq1 probe
  DevBuf force, mass, scratch;
  bool have_force = false, have_mass = false;
  // DEM history (indexed by original id, double-buffered)
  DevBuf hcnt[2], hid[2], hxi[2], wxi[2];
  int cur_hist = 0;
  Timing timing;
  Tape tape;
  bool keep_acc = true;
  // named FP64 fields of generated equations (particle-id order), and the
  // modules compiled for them, keyed by source text
  std::map<std::string, std::unique_ptr<DevBuf>> gfields;
  DevBuf posid;   // positions in id order for the all-pairs form of generated passes
  // read-only model fields bound by generated passes (id-order FP64 copies,
  // refreshed per call), the slot-order copies of [j] fields and the separate
  // outputs of fields a pass reads at [j] and writes, kept between calls
  std::map<std::string, std::unique_ptr<DevBuf>> gmodel, gslots, gsplit;
  struct JitCache {
    std::map<std::string, hipModule_t> mods;
    ~JitCache() {
      for (auto& kv : mods) (void)hipModuleUnload(kv.second);
    }
  } jit;

  // Syncs the stream; throws on a raised flag.  `where` names the stretch of
  // the call the flags cover (e.g. "steps 17-32 of 100").
  void check_flags(const std::string& where = std::string());
};

// Launch helpers -------------------------------------------------------------
constexpr int kBlock = 256;

inline uint32_t blocks_for(uint64_t n, int block = kBlock) {
  return (uint32_t)((n + (uint64_t)block - 1) / (uint64_t)block);
}

// Gather kernels run one wavefront per block over tiles of spatially sorted
// slots, and the hardware deals workgroup b to XCD b % 8.  Block b takes tile
// xcd_tile(b): runs of 32 consecutive tiles per XCD, so that an XCD's L2 keeps
// the neighbour cells its tiles share, while the 8 XCDs move through the
// sorted slots together and tiles of very different cost (a tank's floor and
// top are wall particles only) spread over all of them.  The dispatcher
// balances the rest: a free wavefront slot takes the next block.
//
// Measured against per-XCD ranges of tiles that resident wavefronts claimed
// from device-scope counters (each wavefront probed all eight counters before
// it ended): WCSPH density / force, us: 42,866 particles FP64 79 / 60 -> 67 /
// 52; 200k mixed 120 / 87 -> 105 / 63; 660k FP32 163 / 149 -> 106 / 96; 1.8M
// mixed 329 / 330 -> 285 / 295; 6M FP64 1153 / 1460 -> 1152 / 1335.
constexpr uint32_t kTileRun = 32;
__device__ inline uint32_t xcd_tile(uint32_t b) {
  return b / (8u * kTileRun) * (8u * kTileRun) + (b & 7u) * kTileRun + ((b >> 3) & (kTileRun - 1u));
}
// Blocks that cover n_tiles tiles (the last ones may have none).
inline uint32_t tile_grid(uint32_t n_tiles) { return (n_tiles + 8u * kTileRun - 1u) / (8u * kTileRun) * (8u * kTileRun); }

// Reductions over the wavefront, returned as a wave-uniform value; every lane
// calls.  Row shifts and row broadcasts in the operation itself (its first
// operand through DPP) carry them into lane 63: six instructions and no LDS,
// where shuffles go through the LDS crossbar six times in turn.  The WCSPH
// passes do up to four reductions per run: the FP64 force pass went from 126 to
// 111 registers and from 1362 to 1305 us at 6M particles.
template <class Op>
__device__ inline uint32_t wave_reduce(uint32_t v, uint32_t id, Op&& op) {
  // lanes a control does not reach combine with the identity
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x111, 0xF, 0xF, false));   // row_shr:1
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x112, 0xF, 0xF, false));   // row_shr:2
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x114, 0xF, 0xF, false));   // row_shr:4
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x118, 0xF, 0xF, false));   // row_shr:8
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x142, 0xA, 0xF, false));   // row_bcast:15
  v = op(v, (uint32_t)__builtin_amdgcn_update_dpp((int)id, (int)v, 0x143, 0xC, 0xF, false));   // row_bcast:31
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ inline uint32_t wave_min(uint32_t v) {
  return wave_reduce(v, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return b < a ? b : a; });
}
__device__ inline uint32_t wave_max(uint32_t v) {
  return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return b > a ? b : a; });
}
__device__ inline uint32_t wave_sum(uint32_t v) {
  return wave_reduce(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}

// Maximum of a non-negative float over the wavefront (their bit patterns
// order like the values).
__device__ inline float wave_max_pos(float v) { return __uint_as_float(wave_max(__float_as_uint(v))); }

// Threshold of the FP32 cell scan in units of the cutoff: 1 plus the margin
// that keeps the scan a superset of the exact FP64 test, for offsets up to the
// grid's extent E (in cutoffs) from a wavefront's reference point: 2^-10
// (the test's own rounding) + 16 E 2^-24 (the offsets' rounding).
inline float cell_scan_threshold(const Grid& g, double cutoff) {
  double E = 0.0;
  for (int a = 0; a < 3; ++a) {
    const double lo = g.lo[a], hi = lo + g.dims[a] * g.cs;
    const double e = (std::fabs(lo) > std::fabs(hi) ? std::fabs(lo) : std::fabs(hi)) + (hi - lo);
    E = e > E ? e : E;
  }
  E /= cutoff;
  return (float)(1.0 + 1.0 / 1024.0 + 16.0 * E * 0x1.0p-24);
}

// The FP32 probe's .w carries the particle's cell coordinates modulo 4 (2
// bits per axis: x in bits 6-7, y in 8-9, z in 10-11, bits 0-5 clear).
// Neighbours sit at a cell difference in {-1, 0, 1}, which the residues
// recover exactly: ((c_j - c_i + 1) mod 4) - 1.  With bits 0-5 clear, byte 0
// of w_j - w_i + 64 is ((cx_j - cx_i + 1) mod 4) * 64, which the scan reads
// with a single byte-to-float conversion.
constexpr uint32_t kCodeShift = 6;

__device__ inline uint32_t cell_code(uint32_t cx, uint32_t cy, uint32_t cz) {
  return ((cx & 3u) | ((cy & 3u) << 2) | ((cz & 3u) << 4)) << kCodeShift;
}

__device__ inline int cell_shift(uint32_t wi, uint32_t wj, int axis) {
  const uint32_t s = kCodeShift + 2u * (uint32_t)axis;
  uint32_t t = ((wj >> s) - (wi >> s) + 1u) & 3u;
  return (int)t - 1;
}

// Error message of calls without a context (prestige_last_error(NULL)).
void set_context_free_error(const std::string& msg);

// Copies to and from host memory that is only borrowed for the call; to_host
// waits for the stream (capi.hip).
void to_device(Ctx& c, void* dst, const void* host, size_t bytes);
void to_host(Ctx& c, void* host, const void* src, size_t bytes);

// Per-form kernel entry points (defined in the .hip files).
void neighbors_build(Ctx& c);
MovedOut moved_out(Ctx& c);        // for the next step kernel; its counts then wait for the build
uint64_t sort_tiles(uint64_t n);   // radix-sort tiles of n keys (histogram rows per digit)
void keys_from_positions(Ctx& c);
void eq1_eval(Ctx& c, int loop, double cutoff);
void sph_step_f64(Ctx& c);
void sph_step_f32(Ctx& c);
void sph_step_mixed(Ctx& c);
void sph_density_f64_for_mixed(Ctx& c);   // density of PRESTIGE_FLAG_DENSITY_F64 (FP64 translation unit)
void dem_step_f64(Ctx& c);
void dem_step_mixed(Ctx& c);
void run_equations(Ctx& c, const int32_t* eq_ids, uint32_t n, int32_t loop, double cutoff);
bool generic_field_name(const Ctx& c, const std::string& name);
bool model_field_ids(Ctx& c, const std::string& name, double* d_out);
void scatter_to_ids(Ctx& c, const void* src, int src_kind, int comp, double* d_out);
void gather_from_ids(Ctx& c, const double* d_in, void* dst, int dst_kind, int comp);

}  // namespace prestige
