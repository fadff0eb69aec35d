// emg_internal.h -- context layout and kernel launchers of libemgpu.
// Not part of the public ABI (include/emgpu.h is).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <functional>
#include <string>

#include "emgpu.h"

namespace emg {

constexpr int kBlock = 256;
constexpr int kFixShift = 24;  // rho fixed point: unit CIC weight = 2^24
constexpr double kFixScale = 16777216.0;
constexpr int kJShift = 24;  // current fixed point: 2^24 per unit flux (cell / unit time)
constexpr double kJScale = 16777216.0;
constexpr int kStateSlots = 64;     // saved particle states of the adjoint window
constexpr int kUnsorted = 1 << 30;  // moves_after_sort of a state in no known order

// device error flags
constexpr int kFlagDomain = 1;    // particle outside [0, L] / non-finite
constexpr int kFlagSpillLost = 2; // FP32 re-bucketing lost a particle (capacity)
constexpr int kFlagFar = 4;       // particle moved more than one box length

enum TimerKind { kTPush = 0, kTDeposit = 1, kTSort = 2, kTRelocate = 3, kTEnergy = 4, kTNum = 5 };

struct Grid {
  int nx, ny, nz;
  double slx, sly, slz;
  int cbx, cby;  // FP32 form: bits of ix and iy in the packed cell index (ceil(log2 n))
};

struct SpeciesTab {
  int nspec;
  int64_t off[EMG_MAX_SPECIES + 1];  // segment start in the FP64 state arrays
  int64_t cnt[EMG_MAX_SPECIES];
  double q[EMG_MAX_SPECIES];
  double qm[EMG_MAX_SPECIES];
};

// FP64 (plain) particle state, structure of arrays, species segments at off[]
struct State64 {
  double *x, *y, *z, *vx, *vy, *vz;
  int32_t *pid;
};

// FP32 cell + offset state, structure of arrays, tile-bucketed
struct StateFx {
  int32_t *cell;  // packed ix | iy<<10 | iz<<20
  float *fx, *fy, *fz, *vx, *vy, *vz;
  int32_t *pid;   // nullptr unless the context tracks pid
};

// One mover in a bucket's outbox (32 bytes, two 16-byte halves)
struct alignas(16) FxRec {
  int32_t cell;
  float fx, fy, fz, vx, vy, vz;
  int32_t pid;
};

struct FxBuckets {
  int tile;            // tile edge T
  int ntx, nty, ntz;   // tiles per axis
  int ntiles;          // per species
  int nb;              // nspec * ntiles
  int64_t cap_total;   // slots per buffer (bucket area + spill)
  int64_t area;        // bucket area size (spill region starts here)
  int64_t spill_cap;
  int64_t *start[2];   // [nb + 1] first slot of each bucket
  int32_t *count[2];   // [nb] particles in each bucket
  int32_t *nst[2];     // [nb] of which in the first run (stayers); the rest (direct
                       //      arrivals) sit at the end of the bucket's slots
  int32_t *cap[2];     // [nb] slots owned by each bucket
  int32_t *hist;       // [nb] bucketing scratch: histogram
  int32_t *cursor;     // [nb] bucketing scratch: scatter cursors
  int32_t *spill[2];   // [nspec] spill counters
  int32_t *stay;       // [nb] stayers written by the bucket's workgroup (this step)
  int32_t *extra;      // [nb] direct arrivals reserved by atomics (this step)
  FxRec *ob[2];        // [nb * outbox] movers of each bucket, grouped by direction
  int32_t *pre[2];     // [nb * 28] exclusive prefix of the outbox direction counts
  int32_t *shist[2];   // [nb] spill particles of a buffer, by the bucket of their cell
  int32_t *scur;       // [nb] scatter cursors for them
  int64_t *spre;       // [nb + 1] exclusive prefix of shist
  FxRec *spl;          // [nspec * spill_cap] the spill particles sorted by bucket
  StateFx st[2];
  int cur;             // buffer holding the live particles
  unsigned long long *plan_word;    // [plan blocks] look-back words
  unsigned long long *plan_ticket;  // blocks of plan launches started so far
};

struct Timer {
  hipEvent_t ev[2];
  int pending;
  double total_ms;
  int64_t launches;
  double last_ms;
};

struct EsSolver;  // device field solve (k_poisson.hip)

// Pinned transfer slots of the host read-outs and uploads (emg_io.hip).
constexpr int kIoSlots = 8;
struct HostIo {
  char *pin;
  size_t bytes, stride;
  hipEvent_t ev[kIoSlots];
  bool pending;  // enqueued work still uses the slots
  bool open;     // counted among the process's contexts
};

// An LDS window of the FP64 deposits: nodes o .. o + w - 1 per axis (periodic),
// w <= n, so no node appears twice.
struct Win {
  int32_t wx, wy, wz, ox, oy, oz;
};

struct Cell3 {
  int i, j, k;
};

// most nodes of a window, and the fixed box of a run that no box fits
struct WinShape {
  int cap, fx, fy, fz;
};
// of table 0 (the charge) and 1 (each component of the current), for runs of
// rows or of particles in no order (30 and 3 x 12.8 KB of int64), and for
// patches (12 and 3 x 8 KB: the same margins, two or three nodes)
constexpr WinShape kWinRow[2] = {{3840, 80, 8, 6}, {1600, 40, 8, 5}};
constexpr int kWinPatch[2] = {1536, 1024};
constexpr int kFieldCap = 484;  // field nodes staged by a patch's block: 11 x 11 x 4, 23 KB
static_assert(kWinRow[0].cap % 2 == 0 && kWinRow[1].cap % 2 == 0 && kWinPatch[0] % 2 == 0 &&
                  kWinPatch[1] % 2 == 0, "cleared two entries at a time");

// widen one axis of a window by a node on each side (or to the whole axis) if
// its nodes, times `across` of the other axes, stay within cap
__host__ __device__ inline bool win_grow(int32_t &o, int32_t &w, int n, int across, int cap) {
  if (w >= n || (w + 2 < n ? w + 2 : n) * across > cap) return false;
  if (w + 2 >= n) {
    o = 0;
    w = n;
  } else {
    o = o == 0 ? n - 1 : o - 1;
    w += 2;
  }
  return true;
}

// margins while they fit: z, y, x in turn
__host__ __device__ inline void win_margins(Win &w, const Grid &g, int cap) {
  bool grown = true;
  while (grown) {
    grown = win_grow(w.oz, w.wz, g.nz, w.wx * w.wy, cap);
    grown = win_grow(w.oy, w.wy, g.ny, w.wx * w.wz, cap) || grown;
    grown = win_grow(w.ox, w.wx, g.nx, w.wy * w.wz, cap) || grown;
  }
}

// The window of the cells i .. i + ci - 1, j .. j + cj - 1 of layer k.
__host__ __device__ inline Win patch_window(int i, int j, int k, int ci, int cj, const Grid &g,
                                            int cap) {
  Win w{ci + 1, cj + 1, 2, i, j, k};
  if (w.wx >= g.nx) w.ox = 0, w.wx = g.nx;
  if (w.wy >= g.ny) w.oy = 0, w.wy = g.ny;
  if (w.wz >= g.nz) w.oz = 0, w.wz = g.nz;
  win_margins(w, g, cap);
  return w;
}

// The field nodes staged for the same cells: their own, and one more on each side
// (in z only where that fits) within the nodes 0..n; one node, which serves no
// cell, if even those of the cells are more than cap.
__host__ __device__ inline Win patch_fields(int i, int j, int k, int ci, int cj, const Grid &g,
                                            int cap) {
  Win w{};
  for (int m = 2; m >= 0; m--) {  // margins: x, y, z; x, y; none
    const int mxy = m > 0 ? 1 : 0, mz = m > 1 ? 1 : 0;
    w.ox = i - mxy < 0 ? 0 : i - mxy;
    w.oy = j - mxy < 0 ? 0 : j - mxy;
    w.oz = k - mz < 0 ? 0 : k - mz;
    w.wx = (i + ci + mxy > g.nx ? g.nx : i + ci + mxy) - w.ox + 1;
    w.wy = (j + cj + mxy > g.ny ? g.ny : j + cj + mxy) - w.oy + 1;
    w.wz = (k + 1 + mz > g.nz ? g.nz : k + 1 + mz) - w.oz + 1;
    if (w.wx * w.wy * w.wz <= cap) return w;
  }
  w.wx = w.wy = w.wz = 1;  // a single node: no cell has all its eight
  return w;
}

// The window of a run of rows from cell a to cell b (in the sort order; mid: its middle
// particle's cell).  The cells of a sorted run go from a to b in z-major order
// (rows of the y-z plane one after another), so its nodes fit a box of its rows
// plus one, its layers plus one, and in x the row segment it covers (or, for a
// run that passes into the next row, the periodic range from its first cell to
// its last) or whole rows; the rest of the capacity becomes margins in z, y and
// x for the particles that drift.  A run of more rows than a layer holds, or a
// box over the capacity, gets the fixed box around its middle.
__host__ __device__ inline Win run_window(const Cell3 &a, const Cell3 &b, const Cell3 &mid,
                                          const Grid &g, const WinShape &ws) {
  Win w;
  // the run's rows, as consecutive rows of the periodic y-z plane
  const int64_t plane = (int64_t)g.ny * g.nz;
  int64_t nrow = ((int64_t)b.k * g.ny + b.j) - ((int64_t)a.k * g.ny + a.j) + 1;
  if (nrow <= 0) nrow += plane;
  bool boxed = nrow <= g.ny;
  if (boxed) {
    // x: the row segment a..b, or (a run into the next row) a..nx-1 and 0..b
    // taken as one periodic range; whole rows for longer runs
    w.ox = a.i;
    if (nrow == 1 && b.i >= a.i) w.wx = b.i - a.i + 2;
    else if (nrow == 2 && b.i < a.i) w.wx = b.i + g.nx - a.i + 2;
    else w.wx = g.nx;
    // y: rows a .. b (periodic); z: layers a .. b
    w.oy = a.j;
    w.wy = (int32_t)nrow + 1;
    w.oz = a.k;
    w.wz = (b.k < a.k ? b.k - a.k + g.nz : b.k - a.k) + 2;
    if (w.wx >= g.nx) {
      w.ox = 0;
      w.wx = g.nx;
    }
    if (w.wy >= g.ny) {
      w.oy = 0;
      w.wy = g.ny;
    }
    if (w.wz >= g.nz) {
      w.oz = 0;
      w.wz = g.nz;
    }
    boxed = (int64_t)w.wx * w.wy * w.wz <= ws.cap;
  }
  if (boxed) {
    win_margins(w, g, ws.cap);
  } else {
    w.wx = ws.fx < g.nx ? ws.fx : g.nx;
    w.wy = ws.fy < g.ny ? ws.fy : g.ny;
    w.wz = ws.fz < g.nz ? ws.fz : g.nz;
    auto around = [](int c, int ext, int n) {
      const int v = c - ext / 2;
      return v < 0 ? v + n : v;
    };
    w.ox = around(mid.i, w.wx, g.nx);
    w.oy = around(mid.j, w.wy, g.ny);
    w.oz = around(mid.k, w.wz, g.nz);
  }
  return w;
}

// A block's run of the FP64 kernels after a sort: len consecutive particles
// of species s from its segment's index beg, and their LDS window.
// After a re-sort in patches a run is a patch's particles, cut evenly where
// they are more than kRunMax, or up to kPatchMerge patches of a sparse species.
// After emg_sort each species is cut into blocks of kRunRow particles; a block
// whose particles span fewer than kRunSpan cells is one run, a longer one (a
// sparse region) is cut into np = ceil(span / kRunCells) runs of equal cell
// ranges.  The windows are shaped with the table, once per sort (shaped by
// every block from its particles at every push, the loop was 70% of the scalar
// instructions of the zigzag push and 2-4 us of each block).
struct Run {
  int64_t beg;
  int32_t len, s;
  Win w;
  Win f;  // patches: the field nodes 0..n staged in LDS (not periodic)
};

// The FP64 sort orders, both by z layer first (what the reference's comparator
// asks of spsort): emg_sort's, cells row by row; and that of the library's own
// re-sorts (sort_every), whose layers are cut into patches of kPatch x kPatch
// cells (less at the upper faces), row of patches by row of patches, and each
// patch's cells row by row.  The particles of 64 consecutive cells then reach
// 9 x 9 x 2 nodes instead of 65 x 2 x 2, and drift by less of their window.
constexpr int kPatch = 8;

__host__ __device__ inline int64_t sort_key(int i, int j, int k, const Grid &g, bool patched) {
  if (!patched) return ((int64_t)k * g.ny + j) * g.nx + i;
  const int pj = j / kPatch * kPatch, pi = i / kPatch * kPatch;
  const int h = pj + kPatch <= g.ny ? kPatch : g.ny - pj, w = pi + kPatch <= g.nx ? kPatch : g.nx - pi;
  return ((int64_t)k * g.ny + pj) * g.nx + (int64_t)pi * h + (j - pj) * w + (i - pi);
}

// The sort key of a position: of its cell, each index the int() of the
// coordinate clamped into the grid.
__host__ __device__ inline int64_t sort_key_xyz(double x, double y, double z, const Grid &g,
                                                bool patched) {
  int k = (int)z, j = (int)y, i = (int)x;
  k = k < 0 ? 0 : (k >= g.nz ? g.nz - 1 : k);
  j = j < 0 ? 0 : (j >= g.ny ? g.ny - 1 : j);
  i = i < 0 ? 0 : (i >= g.nx ? g.nx - 1 : i);
  return sort_key(i, j, k, g, patched);
}

// The active lanes of a wave grouped by equal key, one ballot per distinct
// key (no memory access).  Every lane of the wave must call it (the loop is
// uniform).  lead: the group's first lane; inner: the lane's rank in its
// group, in lane order; size: the group's size, on the lead lane.  A caller
// then sends one atomic per group (the lead lane's) instead of one per lane.
__device__ inline void wave_groups(int64_t key, bool act, int &lead, int &inner, int &size) {
  const int lane = __lane_id();
  unsigned long long todo = __ballot(act);
  lead = lane;
  inner = 0;
  size = 0;
  while (todo) {
    const int l = __builtin_amdgcn_readfirstlane(__ffsll((long long)todo) - 1);
    const int64_t k = (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(key >> 32), l)
                                 << 32) |
                                (uint32_t)__builtin_amdgcn_readlane((int)key, l));
    const unsigned long long grp = __ballot(act && key == k);
    if (lane == l) size = __popcll(grp);
    if ((grp >> lane) & 1ull) {
      lead = l;
      inner = __builtin_amdgcn_mbcnt_hi((uint32_t)(grp >> 32),
                                        __builtin_amdgcn_mbcnt_lo((uint32_t)grp, 0));
    }
    todo &= ~grp;
  }
}

// Where a push that carries a re-sort writes particle m of species is: slot
// off[is] + start[is nkey + key] - start[is nkey] + rank[m] of t, key being
// the cell of its position before the move (what sort64_rank counted).
struct SortDest {
  State64 t;
  const int64_t *start;
  const int32_t *rank;
  int64_t nkey;
};

// particles per block of table 0 (charge, ES push) and 1 (zigzag push): of a run
// of rows, or of a slice in no order; and at most of a patch, where a sum of
// kRunMax fixed-point terms of a node still fits (2^48 each; 8 2^48 twice)
constexpr int kRunRow[2] = {4096, 1024};
constexpr int kRunMax[2] = {6144, 2304};
constexpr int kPatchMerge = 4;
constexpr int64_t kRunsUnbuilt = -1;
constexpr int kRunSpan = 96;   // cells a block may span and stay whole
constexpr int kRunCells = 64;  // cells per run of a cut block
static_assert(kRunSpan >= kRunCells, "a cut block's runs span over kRunCells / 2 cells");

// (i, j, k) of point o of an ex x ey x ... box, x fastest; 32-bit divisions
// where they do (a 64-bit one takes about four times the instructions)
__device__ __forceinline__ void point_of(int64_t o, int ex, int ey, int &i, int &j, int &k) {
  if ((o >> 32) == 0) {
    const uint32_t u = (uint32_t)o, q = u / (uint32_t)ex, r = q / (uint32_t)ey;
    i = (int)(u - q * (uint32_t)ex);
    j = (int)(q - r * (uint32_t)ey);
    k = (int)r;
  } else {
    i = (int)(o % ex);
    j = (int)((o / ex) % ey);
    k = (int)(o / ((int64_t)ex * ey));
  }
}

// index modulo n for the indices the grid kernels form (a few cells around
// [0, n)): one compare and add each way, the division only if that misses
__device__ __forceinline__ int periodic_index(int i, int n) {
  int r = i < 0 ? i + n : (i >= n ? i - n : i);
  if ((unsigned)r >= (unsigned)n) r = ((i % n) + n) % n;
  return r;
}

// The device copy of eb: component c of point (i, j, k) at c * np + at(i, j, k).
struct EbView {
  double *eb;
  int lo[3], ext[3];
  int64_t np;
  Grid g;
  __device__ __forceinline__ int64_t at(int i, int j, int k) const {
    return ((int64_t)(k - lo[2]) * ext[1] + (j - lo[1])) * ext[0] + (i - lo[0]);
  }
  // periodic image of cell (i, j, k) inside the stored box
  __device__ __forceinline__ int64_t img(int i, int j, int k) const {
    return at(periodic_index(i, g.nx), periodic_index(j, g.ny), periodic_index(k, g.nz));
  }
};

// Particles binned by tiles (k_bin.hip): counters and cursors per tile, each
// tile's first record, the records of one pass.
constexpr int kBinTile = 8;
struct BinRec {
  double x, y, z;
  int64_t ms;  // the particle's index | species << 56
};
static_assert(sizeof(BinRec) == 32, "two 16-byte accesses");
struct TileBins {
  int32_t *count;
  int64_t *start;
  BinRec *rec;
  int64_t len;  // records
  bool recorded;  // a graph uses them
};
struct BinTiles {
  int ntx, nty, ntz, n;
};

// Upper-face accumulators of the charge.  The periodic accumulators add the
// weight a particle puts on node n of an axis into node 0; the reference
// keeps it apart until its border exchange and add_boundary_charge, which
// leave the raw deposit of node n in ghost plane -1 and that of node 0 in
// plane n + 1.  A face array per species holds the raw weights of the nodes
// with index n on some axis (filled on demand for a read-out of the ghost
// planes): face X = nodes (nx, b, c), b in 0..ny, c in 0..nz; face Y = nodes
// (a, ny, c), a in 0..nx-1, c in 0..nz; face Z = nodes (a, b, nz), a in
// 0..nx-1, b in 0..ny-1.
__host__ __device__ inline int64_t face_len(const Grid &g) {
  return (int64_t)(g.ny + 1) * (g.nz + 1) + (int64_t)g.nx * (g.nz + 1) + (int64_t)g.nx * g.ny;
}

// face slot of node (a, b, c), a in 0..nx, b in 0..ny, c in 0..nz; -1 when no
// index is n
__host__ __device__ inline int64_t face_index(const Grid &g, int a, int b, int c) {
  if (a == g.nx) return (int64_t)c * (g.ny + 1) + b;
  const int64_t y0 = (int64_t)(g.ny + 1) * (g.nz + 1);
  if (b == g.ny) return y0 + (int64_t)c * g.nx + a;
  if (c == g.nz) return y0 + (int64_t)g.nx * (g.nz + 1) + (int64_t)b * g.nx + a;
  return -1;
}

}  // namespace emg

struct emg_ctx {
  emg_config cfg;
  int device;
  hipStream_t stream;
  bool own_stream;
  emg::Grid g;
  int64_t ncell;
  emg::SpeciesTab sp;
  int64_t cap_total;  // FP64: sum of capacities

  // FP64 state
  emg::State64 s64;
  emg::State64 t64;  // sort scratch (lazy)
  bool have_particles;
  int pushes_since_sort;  // PLAIN_FP64 pushes since the last cell sort (sort_every)
  int moves_after_sort;   // PLAIN_FP64 pushes since the state was last sorted, or kUnsorted

  bool ordered;           // the order that was uploaded or loaded keeps neighbours together
  emg::TileBins bins;     // workspace (lazy)

  // FP32 state
  emg::FxBuckets fx;

  // fields
  // eb(6, eb_lo : eb_lo + eb_ext - 1) as six component arrays of eb_points
  // values: an E or a B update writes whole lines, which the six-component
  // records of the boundary's layout would half fill (EbView)
  double *eb_dev;
  size_t eb_dev_bytes;
  bool nodes_b_valid;  // the nodes' B is the relocation of eb_dev's B
  bool b_recorded;     // a graph holds an emg_bfield: its replays change eb_dev's B unseen
  int eb_lo[3], eb_ext[3];
  bool nodes_stale;  // eb changed on the device since the last relocation
  double *fe_buf;    // field-energy partials and result (lazy)
  emg::EsSolver *es; // FFT plans and arrays of the device Poisson solve (lazy)
  double *bk_dev;    // background charge per periodic node (emg_set_background), or null
  double *node64;  // (nx+1)(ny+1)(nz+1) x 8 doubles, nodes 0..n
  float *node32;   // periodic nodes: nx ny nz x (Ex, Ey, Ez, 0), then as many (Bx, By, Bz, 0)
  bool fields_set;

  // deposits
  double *rho64;               // nspec x ncell, q-weighted (FP64 form)
  unsigned long long *rhofx;   // nspec x ncell, unit-weight fixed point
  double *j64;                 // nspec x 3 x ncell, unscaled zigzag sums
  unsigned long long *jfx;     // nspec x 3 x ncell fixed point
  bool rho_valid;
  bool j_valid;
  void *face;       // nspec x face_len: upper-face charge (double, or fixed point in FP32_FIXED)
  // a graph holds a push, and one that moves particles without depositing their
  // charge: its replays move them unseen
  bool push_recorded, move_recorded;
  bool faces_valid; // face holds the deposit of the current positions

  // energy
  double *ke_part;  // partial sums
  int64_t ke_part_n;
  bool ke_valid;

  // sort scratch
  int32_t *sort_count;   // nspec x ncell (or nb)
  int64_t *sort_start;
  int64_t sort_len;
  void *sort_rec;        // cap_total x 64-byte records + cap_total int32 ranks (FP64 sort, lazy)
  emg::Run *runs[2];     // block runs of the last sort: [0] charge, [1] zigzag
  int64_t nruns[2], runs_cap[2];  // (kRunsUnbuilt: not asked for since the last sort)
  int64_t *run_base;     // scan scratch of the run counts (nspec x chunks + 1)
  int64_t run_base_len;
  bool runs_valid;       // the particles are in the order of the sort the runs describe
  bool sort_patched;     // the last sort's order: patches, or emg_sort's rows
  int64_t *scan_tmp;
  int64_t scan_tmp_len;

  int *dflag;       // device error flags, and an upload's count of near neighbours
  int *hflag;       // pinned host mirror
  double *hsum;     // pinned: energies and adjoint sums, written by their kernels
  emg::HostIo io;
  double *scratch;  // this device's static staging array (emg_get_rho_noalloc)

  // adjoint window (FP64 form)
  double *lam;       // 8 per particle slot: lambda_x, lambda_v, 2 unused (one 64-byte line)
  double *adj_e;     // 3 x ncell: transposed gather of qmp * lambda_a
  double *adj_g;     // ncell: uploaded density adjoint
  double *adj_sum;   // block partials of the velocity adjoint sums
  emg::State64 slot[emg::kStateSlots];  // saved particle states
  int64_t slot_cnt[emg::kStateSlots][EMG_MAX_SPECIES];
  bool slot_ordered[emg::kStateSlots];

  bool timing;
  emg::Timer timers[emg::kTNum];
};

namespace emg {

// error plumbing (emg_api.hip)
int set_error(int code, const std::string &msg);
int hip_check(hipError_t e, const char *what);
bool bins_give_back(emg_ctx *c);  // frees bins.rec; false if there is nothing to free

// device memory, the tile records' if there is no other; where there is none a
// null pointer, and no error left for the next launch's check to find
template <typename T>
bool dev_malloc(emg_ctx *c, T **p, size_t bytes) {
  do {
    if (hipMalloc((void **)p, bytes) == hipSuccess) return true;
    (void)hipGetLastError();
  } while (bins_give_back(c));
  *p = nullptr;
  return false;
}

int flags_error(emg_ctx *c);  // *hflag as an error code (and dflag cleared)
bool capturing(emg_ctx *c);   // whether the stream's work is being recorded into a graph

// Host transfers (emg_io.hip) in chunks of whole units.  fill enqueues on the
// context's stream what writes bytes [off, off + len) of the result to the
// pinned slot; io_read copies them to the caller's array and (flags) reports the
// device-side errors first.  use enqueues what reads the slot; the caller's
// array is free when io_write returns.  copy, if given, fills the slot with what
// takes the place of those bytes, at most as many, and returns their number, which
// use gets for len (it is not called for none).  All may be called from several
// threads at once.
using IoFn = std::function<int(size_t off, size_t len, void *slot)>;
using IoCopy = std::function<size_t(size_t off, size_t len, void *slot)>;
int io_read(emg_ctx *c, void *user, size_t bytes, size_t unit, const IoFn &fill, bool flags = true);
int io_write(emg_ctx *c, const void *user, size_t bytes, size_t unit, const IoFn &use,
             const IoCopy &copy = nullptr);
// f(a, b) over ranges that make up [0, n), each entry standing for `bytes` of host
// memory, on the transfers' threads
int io_ranges(emg_ctx *c, int64_t n, size_t bytes,
              const std::function<void(int64_t, int64_t)> &f);
int read_flags(emg_ctx *c);  // synchronise and report device-side errors
// a device array of 8-byte values
int io_read_array(emg_ctx *c, void *user, const void *dev, size_t bytes, bool flags = true);
void io_open(emg_ctx *c);
void io_close(emg_ctx *c);

// timers
void timer_begin(emg_ctx *c, int kind);
void timer_end(emg_ctx *c, int kind);

// scan: exclusive prefix sum of n int32 values into int64 out[0..n]; tmp: scan_tmp_alloc
void exclusive_scan_i32(const int32_t *in, int64_t *out, int64_t n, int64_t *tmp, hipStream_t s);
int scan_tmp_alloc(emg_ctx *c, int64_t n);  // c->scan_tmp for scans of n values

// kernels: FP64 mirror (k_fp64.hip)
void launch_relocate64(emg_ctx *c);  // eb_dev -> the form's nodes
void launch_positn64(emg_ctx *c, int ustep);
// with resort, the push also moves the particles into the order sort64_rank
// has counted (into t64; sort64_commit then makes it the live state)
void launch_push_es64(emg_ctx *c, int ustep, bool resort);
void launch_deposit64(emg_ctx *c);
void launch_push_em64(emg_ctx *c, int ustep, bool resort);
void launch_faces64(emg_ctx *c);  // c->face (zeroed) += upper-face charge
EbView eb_view(const emg_ctx *c);
// device Yee update and field energy on eb_dev (k_yee.hip)
// n points from point o0 on, in the boundary's layout at rec, into eb_dev
void launch_eb_split(emg_ctx *c, const double *rec, int64_t o0, int64_t n);
void launch_bfield(emg_ctx *c);
void launch_efield(emg_ctx *c, double tcs, double dlt);
// points [o0, o0 + n) of the box lo .. lo + ext - 1 (x fastest), 6 values each
void launch_eb_box(emg_ctx *c, const int lo[3], const int ext[3], int64_t o0, int64_t n, double *out);
int64_t field_energy_part_need();
void launch_field_energy(emg_ctx *c, double cs, double *part_dev, double *out);
// device ES field solve (k_poisson.hip): rho of the last deposit + rhobk ->
// phi -> E into eb_dev -> nodes
int solve_es(emg_ctx *c, double rhobk);
int read_potential(emg_ctx *c, double *phi);
int es_solver_stream(emg_ctx *c);  // after c->stream has changed
void es_solver_free(emg_ctx *c);

// common kernels (k_common.hip)
// energy sums (3 per species) into hsum, and the device flags into hflag
void launch_energy64(emg_ctx *c);
// points [o0, o0 + n) of a read-out of lo..hi into dst; prepare_read_rho first:
// true if the box holds ghost planes, whose charge it then deposits
bool prepare_read_rho(emg_ctx *c, const int lo[3], const int hi[3]);
void launch_read_rho(emg_ctx *c, int species, bool ghosts, double *dst, const int lo[3],
                     const int hi[3], int64_t o0, int64_t n);
void launch_read_current(emg_ctx *c, int species, double *dst, const int lo[3], const int hi[3],
                         int64_t o0, int64_t n);
void launch_zero(void *p, size_t bytes, hipStream_t s);
// The FP64 cell sort.  sort64 sorts the live state.  A re-sort close to the
// last sort can ride on the next push instead: sort64_rank counts the
// current cells (each key's start, each particle's rank in its key), the
// push writes every particle to its sorted slot (SortDest), and sort64_commit
// makes that the live state.  A run table is built when a launch first needs it.
int sort64(emg_ctx *c, bool patched);
int sort64_runs(emg_ctx *c, int which);  // the run table of the charge (0) or the zigzag (1)
bool sort64_fusable(const emg_ctx *c);
int sort64_rank(emg_ctx *c, int which);  // which: the run table of the push that follows
SortDest sort64_dest(const emg_ctx *c);
int sort64_commit(emg_ctx *c);
int init_device(emg_ctx *c, const emg_device_species *spec, int nspec, uint64_t seed);

// binning by tiles (k_bin.hip): bin_pass bins the next particles of every
// species, after done[] of it, into bins.rec and bins.start, and returns how
// many (0: none left)
BinTiles bin_tiles(const Grid &g);
int bins_alloc(emg_ctx *c);
int64_t bin_pass(emg_ctx *c, int64_t done[EMG_MAX_SPECIES]);

// adjoint of the FP64 ES push (k_adj.hip)
void launch_adj_step64(emg_ctx *c, int ustep);  // after bins_alloc
void launch_adj_density64(emg_ctx *c, const double *qfac);  // one factor per species
void launch_adj_vsum(emg_ctx *c, double *part, double *out);  // part: adj_vsum_need() doubles
int64_t adj_vsum_need();

// FP32 + fixed point (k_fx.hip)
int fx_alloc(emg_ctx *c, int64_t ntotal);
int fx_from64(emg_ctx *c, const State64 &src);       // convert + bucket
int fx_to64(emg_ctx *c, State64 &dst);               // convert back (species contiguous)
void launch_fx_step(emg_ctx *c, int ustep, bool push, bool deposit, bool em);
void launch_fx_deposit(emg_ctx *c);
void launch_fx_energy(emg_ctx *c);
void launch_fx_faces(emg_ctx *c);  // c->face (zeroed) += upper-face charge, fixed point
void fx_energy_from_push(emg_ctx *c);
int fx_rebucket(emg_ctx *c);

}  // namespace emg
