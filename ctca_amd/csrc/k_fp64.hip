// k_fp64.hip -- plain FP64 kernels of the particle path: the drop-in form that
// mirrors the reference arithmetic operation by operation.  Compiled with
// -ffp-contract=off, so every multiply and add is rounded separately in the
// reference's source order (and so bit-identical to a CPU restatement built the
// same way).  One thread per particle, species segments on blockIdx.y, state
// in place (structure of arrays), deposition with FP64 global atomics into
// periodic accumulators (node index mod n == the single-rank fold).
#include <algorithm>

#include "emg_internal.h"

namespace emg {
namespace {

__device__ __forceinline__ int64_t nidx64(const Grid &g, int i, int j, int k) {
  // nodal FP64 field, nodes 0..n per axis
  return ((int64_t)k * (g.ny + 1) + j) * (g.nx + 1) + i;
}

__device__ __forceinline__ int wrapn(int i, int n) {
  // node / cell index in [-n, 2n) -> [0, n)
  return i < 0 ? i + n : (i >= n ? i - n : i);
}

__device__ __forceinline__ int64_t cidx(const Grid &g, int i, int j, int k) {
  return ((int64_t)wrapn(k, g.nz) * g.ny + wrapn(j, g.ny)) * g.nx + wrapn(i, g.nx);
}

// Guard against positions the reference would index out of bounds with:
// anything outside [0, L] or non-finite is clamped and reported.
__device__ __forceinline__ void domain_guard(double &x, double &y, double &z, const Grid &g,
                                             int *flag) {
  bool ok = (x >= 0.0) && (x <= g.slx) && (y >= 0.0) && (y <= g.sly) && (z >= 0.0) &&
            (z <= g.slz);
  if (!ok) {
    atomicOr(flag, kFlagDomain);
    x = (x >= 0.0) ? (x <= g.slx ? x : g.slx) : 0.0;
    y = (y >= 0.0) ? (y <= g.sly ? y : g.sly) : 0.0;
    z = (z >= 0.0) ? (z <= g.slz ? z : g.slz) : 0.0;
  }
}

struct Cic {
  double v1, v2, v3, v4, v5, v6, v7, v8;
  int i, j, k;
};

// CIC weights, src/pcl2field/psolve2.F90:154-183 (charge.F90:160-193).
// xl, yl, zl are the cell-local coordinates, i/j/k the already truncated cell.
__device__ __forceinline__ Cic cic(double xl, double yl, double zl, int i, int j, int k) {
  Cic w;
  w.i = i;
  w.j = j;
  w.k = k;
  double x1 = xl - (double)i, y1 = yl - (double)j, z1 = zl - (double)k;
  double xy1 = x1 * y1, xz1 = x1 * z1, yz1 = y1 * z1;
  double z2 = 1.0 - z1;
  double xz2 = x1 * z2, yz2 = y1 * z2;
  w.v3 = xy1 * z1;
  w.v2 = xz1 - w.v3;
  w.v4 = yz1 - w.v3;
  w.v1 = z1 - xz1 - w.v4;
  w.v7 = xy1 * z2;
  w.v6 = xz2 - w.v7;
  w.v8 = yz2 - w.v7;
  w.v5 = z2 - xz2 - w.v8;
  return w;
}

// the two nodes of a row (x edge), six components each
struct Row {
  double a[6], b[6];
};
__device__ __forceinline__ Row load_row(const double *p, int dx) {
  const double2 *q = reinterpret_cast<const double2 *>(p);
  const double2 *r = reinterpret_cast<const double2 *>(p + dx);
  const double2 a = q[0], b = q[1], c = q[2], d = r[0], e = r[1], f = r[2];
  return {{a.x, a.y, b.x, b.y, c.x, c.y}, {d.x, d.y, e.x, e.y, f.x, f.y}};
}

// psolve2.F90:195-218: eight-node gather of the six nodal components in the
// reference's node order v1..v8 and summation order, a row at a time: left to
// itself the compiler has all eight nodes (96 registers) in flight.  DEEP
// keeps two rows in flight, the charge push's 124 VGPRs holding four waves per
// SIMD; else one row, with which the zigzag push fits 128 and holds four waves
// instead of three (128^3 charge push 8.41 -> 8.33 ms with DEEP; zigzag push
// of 18.5M particles 1.42 -> 1.33 ms without).
template <bool DEEP>
__device__ __forceinline__ void gather6(const double *__restrict__ node, const Grid &g,
                                        const Cic &w, double f[6]) {
  const double *p = node + 8 * nidx64(g, w.i, w.j, w.k);
  const int dx = w.i < g.nx ? 8 : 0;
  const int64_t dj = w.j < g.ny ? 8 * (int64_t)(g.nx + 1) : 0;
  const int64_t dk = w.k < g.nz ? 8 * (int64_t)(g.nx + 1) * (g.ny + 1) : 0;
if (DEEP) {
    const Row r1 = load_row(p + dk, dx);
    const Row r2 = load_row(p + dk + dj, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = r1.a[c] * w.v1 + r1.b[c] * w.v2;
    const Row r3 = load_row(p + 0, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r2.b[c] * w.v3 + r2.a[c] * w.v4;
    const Row r4 = load_row(p + dj, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r3.a[c] * w.v5 + r3.b[c] * w.v6;
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r4.b[c] * w.v7 + r4.a[c] * w.v8;
  } else {
    const Row r1 = load_row(p + dk, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = r1.a[c] * w.v1 + r1.b[c] * w.v2;
    const Row r2 = load_row(p + dk + dj, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r2.b[c] * w.v3 + r2.a[c] * w.v4;
    const Row r3 = load_row(p + 0, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r3.a[c] * w.v5 + r3.b[c] * w.v6;
    const Row r4 = load_row(p + dj, dx);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 6; c++) f[c] = f[c] + r4.b[c] * w.v7 + r4.a[c] * w.v8;
  }
}

// The same from the block's staged nodes fs (three double2 per node, box F),
// for a cell whose eight nodes are among them.
__device__ __forceinline__ bool staged(const Win &F, const Cic &w) {
  return (unsigned)(w.i - F.ox) < (unsigned)(F.wx - 1) &&
         (unsigned)(w.j - F.oy) < (unsigned)(F.wy - 1) &&
         (unsigned)(w.k - F.oz) < (unsigned)(F.wz - 1);
}

__device__ __forceinline__ void gather6_lds(const double2 *fs, const Win &F, const Cic &w,
                                            double f[6]) {
  const double2 *p = fs + 3 * (((w.k - F.oz) * F.wy + (w.j - F.oy)) * F.wx + (w.i - F.ox));
  const int dj = 3 * F.wx, dk = dj * F.wy;
  auto row = [](const double2 *q) {
    const double2 a = q[0], b = q[1], c = q[2], d = q[3], e = q[4], g = q[5];
    return Row{{a.x, a.y, b.x, b.y, c.x, c.y}, {d.x, d.y, e.x, e.y, g.x, g.y}};
  };
  const Row r1 = row(p + dk), r2 = row(p + dk + dj);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 6; c++) f[c] = r1.a[c] * w.v1 + r1.b[c] * w.v2;
  const Row r3 = row(p);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 6; c++) f[c] = f[c] + r2.b[c] * w.v3 + r2.a[c] * w.v4;
  const Row r4 = row(p + dj);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int c = 0; c < 6; c++) f[c] = f[c] + r3.a[c] * w.v5 + r3.b[c] * w.v6;
#pragma unroll
  for (int c = 0; c < 6; c++) f[c] = f[c] + r4.b[c] * w.v7 + r4.a[c] * w.v8;
}

__device__ __forceinline__ void stage_fields(double2 *fs, const Win &F,
                                             const double *__restrict__ node, const Grid &g) {
  const int n = 3 * F.wx * F.wy * F.wz;
  for (int q = threadIdx.x; q < n; q += blockDim.x) {
    const int v = q / 3, r = v / F.wx;
    const int k = r / F.wy;
    const double *p = node + 8 * nidx64(g, F.ox + v - r * F.wx, F.oy + r - k * F.wy, F.oz + k);
    fs[q] = reinterpret_cast<const double2 *>(p)[q - 3 * v];
  }
}

// Buneman-Boris, psolve2.F90:233-257 (ewmodel = 0: the wave field is +0.0).
__device__ __forceinline__ void boris64(double &vx, double &vy, double &vz, const double f[6],
                                        double qmp) {
  const double ewx = 0.0, ewy = 0.0;
  double eex = (f[0] + ewx) * qmp;
  double eey = (f[1] + ewy) * qmp;
  double eez = f[2] * qmp;
  double bbx = f[3] * qmp, bby = f[4] * qmp, bbz = f[5] * qmp;
  double bor = 2.0 / (1.0 + bbx * bbx + bby * bby + bbz * bbz);
  vx = vx + eex;
  vy = vy + eey;
  vz = vz + eez;
  double vxt = vx + vy * bbz - vz * bby;
  double vyt = vy + vz * bbx - vx * bbz;
  double vzt = vz + vx * bby - vy * bbx;
  vx = vx + bor * (vyt * bbz - vzt * bby);
  vy = vy + bor * (vzt * bbx - vxt * bbz);
  vz = vz + bor * (vxt * bby - vyt * bbx);
  vx = vx + eex;
  vy = vy + eey;
  vz = vz + eez;
}

// psolve2.F90:354-432 / positn.F90:172-254, npbnd = 0: one wrap per axis
__device__ __forceinline__ void wrap_periodic(double &x, double &y, double &z, const Grid &g,
                                              int *flag) {
  if (x < 0.0 || x >= g.slx || y < 0.0 || y >= g.sly || z < 0.0 || z >= g.slz) {
    if (x < 0.0) x = x + g.slx; else if (x >= g.slx) x = x - g.slx;
    if (y < 0.0) y = y + g.sly; else if (y >= g.sly) y = y - g.sly;
    if (z < 0.0) z = z + g.slz; else if (z >= g.slz) z = z - g.slz;
    if (!(x >= 0.0 && x <= g.slx && y >= 0.0 && y <= g.sly && z >= 0.0 && z <= g.slz))
      atomicOr(flag, kFlagFar);
  }
}

// ---------------------------------------------------------------- grdcrt
// grdcrt.F90:158-169 (E) and 216-230 (B); writes nodes 0..n in FP64 (node64) or
// the periodic nodes 0..n-1 in FP32 (node32) of the same values.
__global__ __launch_bounds__(kBlock) void k_relocate(EbView v, double *__restrict__ node64,
                                                     float *__restrict__ node32, int64_t ncell,
                                                     double e0x, double e0y, double e0z,
                                                     double b0x, double b0y, double b0z) {
  const Grid &g = v.g;
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t nn = (int64_t)(g.nx + 1) * (g.ny + 1) * (g.nz + 1);
  if (idx >= nn) return;
  int i, j, k;
  point_of(idx, g.nx + 1, g.ny + 1, i, j, k);
  if (node32 && (i == g.nx || j == g.ny || k == g.nz)) return;
  const double *p = v.eb + v.at(i, j, k);
  const int64_t np = v.np, sy = v.ext[0], sz = (int64_t)v.ext[0] * v.ext[1];
  const double *ex = p, *ey = p + np, *ez = p + 2 * np, *bx = p + 3 * np, *by = p + 4 * np,
               *bz = p + 5 * np;
  double o[6];
  o[0] = 0.5 * (ex[0] + ex[-1]) + e0x;
  o[1] = 0.5 * (ey[0] + ey[-sy]) + e0y;
  o[2] = 0.5 * (ez[0] + ez[-sz]) + e0z;
  o[3] = 0.25 * (bx[0] + bx[-sy] + bx[-sz] + bx[-sy - sz]) + b0x;
  o[4] = 0.25 * (by[0] + by[-1] + by[-sz] + by[-1 - sz]) + b0y;
  o[5] = 0.25 * (bz[0] + bz[-1] + bz[-sy] + bz[-1 - sy]) + b0z;
  if (node64) {
    double2 *d = reinterpret_cast<double2 *>(node64 + 8 * idx);
    d[0] = make_double2(o[0], o[1]);
    d[1] = make_double2(o[2], o[3]);
    d[2] = make_double2(o[4], o[5]);
    d[3] = make_double2(0.0, 0.0);
  }
  if (node32) {
    const int64_t c = ((int64_t)k * g.ny + j) * g.nx + i;
    float4 *d = reinterpret_cast<float4 *>(node32);
    d[c] = make_float4((float)o[0], (float)o[1], (float)o[2], 0.f);
    d[ncell + c] = make_float4((float)o[3], (float)o[4], (float)o[5], 0.f);
  }
}

// ---------------------------------------------------------------- positn
__global__ __launch_bounds__(kBlock) void k_positn64(State64 s, SpeciesTab sp, Grid g, int ustep,
                                                     int *flag) {
  int is = blockIdx.y;
  int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= sp.cnt[is]) return;
  m += sp.off[is];
  double us = (double)ustep;
  double x = s.x[m], y = s.y[m], z = s.z[m];
  x = x + s.vx[m] * us;
  y = y + s.vy[m] * us;
  z = z + s.vz[m] * us;
  wrap_periodic(x, y, z, g, flag);
  s.x[m] = x;
  s.y[m] = y;
  s.z[m] = z;
}

// ---------------------------------------------------------------- psolve2 + charge
// ---------------------------------------------------------------- charge
// charge.F90:59-83 + distribute_charge 197-210; rho[is][node mod n] += v_k q(is)
// charge.F90:152-210 per particle; the particles of a block are a contiguous
// run of a species.  The sort orders particles by cell and they drift slowly,
// so most of a block's particles lie in a box of nodes: the block sums their
// weights in an LDS window of that box, as int64 fixed point at 2^48 per unit
// weight (at most kRunMax[0] terms of at most 2^48 per node, below 2^61), and
// adds each non-zero window node
// times q(is) to rho with one global FP64 atomic; a particle whose eight
// nodes are not all in the window adds its weights to rho directly.  The
// rounding of a weight (2^-49) is below the FP64 round-off of the sequential
// sum, which the reference's order would give.  The block's particles and its
// window: block_run.
constexpr double kRhoFix = 281474976710656.0;   // 2^48 per unit weight

// window index of node l + 1 on an axis of window extent w (full axis: w = n,
// where node n is node 0); false if it is outside the window
__device__ __forceinline__ bool win_next(int l, int w, int n, int &l1) {
  l1 = l + 1;
  if (l1 < w) return true;
  l1 = 0;
  return w == n && l + 1 == n;
}

// The window of particles a .. b of no run table: from the cells of the first,
// the last and the middle one.
__device__ __forceinline__ Win slice_window(const State64 &s, int64_t a, int64_t b, const Grid &g,
                                            const WinShape &ws) {
  auto cell = [&](int64_t m) {
    const double x = s.x[m], y = s.y[m], z = s.z[m];
    return Cell3{min(max((int)x, 0), g.nx - 1), min(max((int)y, 0), g.ny - 1),
                 min(max((int)z, 0), g.nz - 1)};
  };
  return run_window(cell(a), cell(b), cell(a + (b - a) / 2), g, ws);
}

// The block's run of particles (indices in the species' segment) and its
// window: after a sort the run table's entry (at most `per` particles over a
// bounded range of cells), else the per-th slice of species blockIdx.y.  False
// for a block past the end.
__device__ __forceinline__ bool block_run(const State64 &s, const SpeciesTab &sp, const Run *runs,
                                          int per, const Grid &g, const WinShape &ws, int &is,
                                          int64_t &beg, int64_t &end, Win &W, Win &F) {
  if (runs) {
    const Run r = runs[blockIdx.x];
    if (r.len == 0) return false;
    is = r.s;
    beg = r.beg;
    end = r.beg + r.len;
    W = r.w;
    F = r.f;
    return true;
  }
  is = blockIdx.y;
  beg = (int64_t)blockIdx.x * per;
  const int64_t cnt = sp.cnt[is];
  if (beg >= cnt) return false;
  end = min(beg + (int64_t)per, cnt);
  W = slice_window(s, sp.off[is] + beg, sp.off[is] + end - 1, g, ws);
  return true;
}

// v times 2^48 rounded to the nearest integer, |v| < 8: the sum with 1.5 2^52
// has an ulp of 1, so its mantissa holds the integer; 1.5 2^52 has a zero low
// word, so taking it off is one 32-bit subtraction (a conversion to int64 is
// about seven instructions)
__device__ __forceinline__ unsigned long long win_fix(double v) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(
      __builtin_fma(v, 281474976710656.0, 6755399441055744.0));
  return ((unsigned long long)((uint32_t)(b >> 32) - 0x43380000u) << 32) | (uint32_t)b;
}

// One particle's CIC weights (charge.F90:152-210) at (x, y, z): into the
// block's LDS window when its eight nodes lie in it, else into the species'
// rho r directly.
__device__ __forceinline__ void deposit_win(unsigned long long *win, const Win &W, double *r,
                                            const Grid &g, double x, double y, double z,
                                            double qc) {
  int i = (int)x, j = (int)y, k = (int)z;
  Cic w = cic(x, y, z, i, j, k);
  // window coordinates of the cell (cell n, of a position at L, is cell 0's image)
  int li = wrapn(i - W.ox + g.nx, g.nx), lj = wrapn(j - W.oy + g.ny, g.ny),
      lk = wrapn(k - W.oz + g.nz, g.nz);
  int li1, lj1, lk1;
  if (li < W.wx && lj < W.wy && lk < W.wz && win_next(li, W.wx, g.nx, li1) &&
      win_next(lj, W.wy, g.ny, lj1) && win_next(lk, W.wz, g.nz, lk1)) {
    auto at = [&](int a, int b, int c) { return win + (c * W.wy + b) * W.wx + a; };
    atomicAdd(at(li, lj, lk1), win_fix(w.v1));
    atomicAdd(at(li1, lj, lk1), win_fix(w.v2));
    atomicAdd(at(li1, lj1, lk1), win_fix(w.v3));
    atomicAdd(at(li, lj1, lk1), win_fix(w.v4));
    atomicAdd(at(li, lj, lk), win_fix(w.v5));
    atomicAdd(at(li1, lj, lk), win_fix(w.v6));
    atomicAdd(at(li1, lj1, lk), win_fix(w.v7));
    atomicAdd(at(li, lj1, lk), win_fix(w.v8));
  } else {
    int i1 = i + 1, j1 = j + 1, k1 = k + 1;
    atomicAdd(r + cidx(g, i, j, k1), w.v1 * qc);
    atomicAdd(r + cidx(g, i1, j, k1), w.v2 * qc);
    atomicAdd(r + cidx(g, i1, j1, k1), w.v3 * qc);
    atomicAdd(r + cidx(g, i, j1, k1), w.v4 * qc);
    atomicAdd(r + cidx(g, i, j, k), w.v5 * qc);
    atomicAdd(r + cidx(g, i1, j, k), w.v6 * qc);
    atomicAdd(r + cidx(g, i1, j1, k), w.v7 * qc);
    atomicAdd(r + cidx(g, i, j1, k), w.v8 * qc);
  }
}

// The window's non-zero nodes into the C accumulators r[0..C-1] (sums times
// scale), one FP64 atomic each, after a barrier; component c of the window
// starts at c * nodes.  The thread's node moves on by kBlock per pass: its
// three indices are carried along (four integer divisions per node and
// component, as many VALU instructions as half of the zigzag push's particle
// work, were 20% of that kernel's time).
template <int C>
__device__ __forceinline__ void flush_win(const unsigned long long *win, const Win &W,
                                          double *const r[C], const Grid &g, double scale) {
  const int nodes = W.wx * W.wy * W.wz;
  int q = threadIdx.x;
  const int t = q / W.wx, st = kBlock / W.wx;
  int li = q - t * W.wx, lk = t / W.wy, lj = t - lk * W.wy;
  const int sx = kBlock - st * W.wx, sz = st / W.wy, sy = st - sz * W.wy;
  for (; q < nodes; q += kBlock) {
    long long v[C];
    bool any = false;
#pragma unroll
    for (int c = 0; c < C; c++) {
      v[c] = (long long)win[c * nodes + q];
      any = any || v[c] != 0;
    }
    if (any) {
      const int64_t n = cidx(g, W.ox + li, W.oy + lj, W.oz + lk);
#pragma unroll
      for (int c = 0; c < C; c++)
        if (v[c] != 0) atomicAdd(r[c] + n, (double)v[c] * scale);
    }
    li += sx;
    lj += sy;
    lk += sz;
    if (li >= W.wx) {
      li -= W.wx;
      lj++;
    }
    if (lj >= W.wy) {
      lj -= W.wy;
      lk++;
    }
  }
}

// clear the first n of an even number of window entries
__device__ __forceinline__ void zero_win(unsigned long long *win, int n) {
  for (int q = threadIdx.x; 2 * q < n; q += blockDim.x)
    reinterpret_cast<ulonglong2 *>(win)[q] = make_ulonglong2(0ull, 0ull);
}

__global__ __launch_bounds__(kBlock) void k_deposit64(State64 s, SpeciesTab sp, Grid g,
                                                      double *__restrict__ rho, int64_t ncell,
                                                      const Run *__restrict__ runs, int *flag) {
  extern __shared__ __align__(16) unsigned long long win[];
  int is;
  int64_t beg, end;
  Win W, F;
  if (!block_run(s, sp, runs, kRunRow[0], g, kWinRow[0], is, beg, end, W, F)) return;  // uniform
  const int64_t off = sp.off[is];
  zero_win(win, W.wx * W.wy * W.wz);
  __syncthreads();
  const double qc = sp.q[is];
  double *r = rho + (int64_t)is * ncell;
  for (int64_t m = beg + threadIdx.x; m < end; m += kBlock) {
    double x = s.x[off + m], y = s.y[off + m], z = s.z[off + m];
    domain_guard(x, y, z, g, flag);
    deposit_win(win, W, r, g, x, y, z, qc);
  }
  __syncthreads();
  double *const acc[1] = {r};
  flush_win<1>(win, W, acc, g, qc / kRhoFix);
}

// The charge of an unsorted state, binned by tiles (k_bin.hip): one workgroup
// per tile and slice adds its records' weights in FP64 LDS tiles, one per
// species, whose nodes reach rho once (a node strictly inside a tile that one
// workgroup does: without an atomic).  Particle by particle into rho, the eight
// atomics of 46 ps each were all of the time: 1.77M particles on 48^3 cells 654
// us with the push; 151 (push) + 126 (binning) + 19 us this way.
constexpr int kTileBlock = 512;
constexpr int kTileNodes = (kBinTile + 1) * (kBinTile + 1) * (kBinTile + 1);

__global__ __launch_bounds__(kTileBlock) void k_tile_charge(const BinRec *__restrict__ rec,
                                                           const int64_t *__restrict__ start,
                                                           BinTiles at, SpeciesTab sp, Grid g,
                                                           double *__restrict__ rho, int64_t ncell,
                                                           int *flag) {
  extern __shared__ double tile[];  // nspec x kTileNodes
  constexpr int N = kBinTile + 1;
  const int tl = blockIdx.x;
  const int64_t beg = start[tl], end = start[tl + 1];
  const int64_t step = (int64_t)gridDim.y * kTileBlock;
  if (beg + (int64_t)blockIdx.y * kTileBlock >= end) return;  // uniform over the block
  const int ox = (tl % at.ntx) * kBinTile, oy = (tl / at.ntx) % at.nty * kBinTile,
            oz = tl / (at.ntx * at.nty) * kBinTile;
  for (int q = threadIdx.x; q < sp.nspec * kTileNodes; q += kTileBlock) tile[q] = 0.0;
  __syncthreads();
  for (int64_t m = beg + (int64_t)blockIdx.y * kTileBlock + threadIdx.x; m < end; m += step) {
    const double2 *r = reinterpret_cast<const double2 *>(rec + m);
    const double2 r0 = r[0], r1 = r[1];
    double x = r0.x, y = r0.y, z = r1.x;
    domain_guard(x, y, z, g, flag);
    const int i = min((int)x, g.nx - 1), j = min((int)y, g.ny - 1), k = min((int)z, g.nz - 1);
    const Cic w = cic(x, y, z, i, j, k);
    double *p = tile + (int)(__double_as_longlong(r1.y) >> 56) * kTileNodes +
                ((k - oz) * N + (j - oy)) * N + (i - ox);
    atomicAdd(p + N * N, w.v1);
    atomicAdd(p + N * N + 1, w.v2);
    atomicAdd(p + N * N + N + 1, w.v3);
    atomicAdd(p + N * N + N, w.v4);
    atomicAdd(p, w.v5);
    atomicAdd(p + 1, w.v6);
    atomicAdd(p + N + 1, w.v7);
    atomicAdd(p + N, w.v8);
  }
  __syncthreads();
  const int tx = min(kBinTile, g.nx - ox), ty = min(kBinTile, g.ny - oy),
            tz = min(kBinTile, g.nz - oz);
  for (int q = threadIdx.x; q < sp.nspec * kTileNodes; q += kTileBlock) {
    const int s = q / kTileNodes, v = q - s * kTileNodes;
    const int i = v % N, j = (v / N) % N, k = v / (N * N);
    const double t = tile[q] * sp.q[s];
    if (i > tx || j > ty || k > tz || t == 0.0) continue;
    double *d = rho + s * ncell + cidx(g, ox + i, oy + j, oz + k);
    if (gridDim.y == 1 && i > 0 && i < tx && j > 0 && j < ty && k > 0 && k < tz) *d += t;
    else atomicAdd(d, t);
  }
}

// psolve2 and charge in one pass (psolve2.F90:137-433, then charge.F90:
// 59-83): each particle of the block's run is pushed with the reference's
// arithmetic in its order -- int() cell, CIC weights, eight-node gather,
// Buneman-Boris, x += v ustep, periodic wrap -- and its charge deposited at
// the new position exactly as k_deposit64 would.
// The window is shaped from the run's positions before the move (read by
// every thread before any is written: the barrier after zeroing it); the
// particles that move out of it add to rho directly.
// RESORT: the moved particle (and its pid) goes to its sorted slot of dst.t
// instead of back to its own slot; the arithmetic is the same.  Four waves
// per SIMD (at most 128 VGPRs) for both forms: the plain one needs 122, the
// re-sorting one would take 132 and drop to three.
// STAGED (runs of patches): the patch's field nodes are copied to LDS first and
// the gather reads them there.  From memory it moves 24 x 16 bytes per particle
// through the vector cache, 384 of its cycles per wave and round, whatever the
// lanes share.  On 128^3 cells with 64 particles per cell and species, per step
// with the re-sorts: rows 8.31 ms, patches 8.73, patches with staged fields
// 7.49; 64^3 with 16 per cell 426, 408 and 327 us.
// DEP = false (an unsorted state): no charge, launch_tiles64 deposits it.
template <bool RESORT, bool STAGED, bool DEP = true>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
void k_push_dep64(State64 s, SpeciesTab sp, const double *__restrict__ node, Grid g, int ustep,
                  double *__restrict__ rho, int64_t ncell, const Run *__restrict__ runs, int *flag,
                  SortDest dst) {
  extern __shared__ __align__(16) unsigned long long win[];
  int is;
  int64_t beg, end;
  Win W, F;
  if (!block_run(s, sp, runs, kRunRow[0], g, kWinRow[0], is, beg, end, W, F)) return;  // uniform
  const int64_t off = sp.off[is];
  const int64_t key0 = (int64_t)is * dst.nkey;
  const int64_t base = RESORT ? off - dst.start[key0] : 0;
  double2 *fs = reinterpret_cast<double2 *>(win + kWinPatch[0]);
  if (DEP) zero_win(win, W.wx * W.wy * W.wz);
  if (STAGED) stage_fields(fs, F, node, g);
  __syncthreads();
  const double gustep = (double)ustep;
  const double qmp = sp.qm[is] * gustep * 0.5;
  const double qc = sp.q[is];
  double *r = rho + (int64_t)is * ncell;
  for (int64_t mm = beg + threadIdx.x; mm < end; mm += kBlock) {
    const int64_t m = off + mm;
    double x = s.x[m], y = s.y[m], z = s.z[m];
    double vx = s.vx[m], vy = s.vy[m], vz = s.vz[m];
    int64_t d = m;
    int32_t pid = 0;
    if (RESORT) {
      pid = s.pid[m];
      d = base + dst.start[key0 + sort_key_xyz(x, y, z, g, true)] + dst.rank[m];
    }
    domain_guard(x, y, z, g, flag);
    int i = (int)x, j = (int)y, k = (int)z;  // int(), psolve2.F90:158-160
    Cic w = cic(x, y, z, i, j, k);
    double f[6];
    if (STAGED && staged(F, w)) gather6_lds(fs, F, w, f);
    else gather6<!STAGED>(node, g, w, f);
    boris64(vx, vy, vz, f, qmp);
    double xmove = vx * gustep, ymove = vy * gustep, zmove = vz * gustep;
    x = x + xmove;
    y = y + ymove;
    z = z + zmove;
    wrap_periodic(x, y, z, g, flag);
    const State64 &o = RESORT ? dst.t : s;
    o.x[d] = x;
    o.y[d] = y;
    o.z[d] = z;
    o.vx[d] = vx;
    o.vy[d] = vy;
    o.vz[d] = vz;
    if (RESORT) o.pid[d] = pid;
    if (DEP) {
      domain_guard(x, y, z, g, flag);
      deposit_win(win, W, r, g, x, y, z, qc);
    }
  }
  if (!DEP) return;
  __syncthreads();
  double *const acc[1] = {r};
  flush_win<1>(win, W, acc, g, qc / kRhoFix);
}

// ---------------------------------------------------------------- psolve1
// psolve1.F90:146-789: push with floor() cells, then the Umeda zigzag current
// of the two segments b -> relay -> a; J[is][c][cell mod n] += vv * w (q(is)
// is applied at read-out, psolve1.F90:793-802).
struct Relay {
  double la, a, r;
  int ia;
};

__device__ __forceinline__ Relay relay_axis(double xnew, double lb, double cb, int ib, int n,
                                            double sl, bool inside, double &pos) {
  Relay r;
  if (!inside && xnew < 0.0) {  // psolve1.F90:440-447
    r.la = xnew;
    pos = xnew + sl;
    r.ia = -1;
    r.a = -1.0;
    r.r = 0.0;
  } else if (!inside && xnew >= sl) {  // :462-469
    r.la = xnew - 0.0;
    pos = xnew - sl;
    r.ia = n;
    r.a = (double)n;
    r.r = (double)n;
  } else {  // :381-415, :469-478
    r.la = xnew - 0.0;
    pos = xnew;
    r.ia = (int)floor(r.la);
    r.a = (double)r.ia;
    r.r = (ib == r.ia) ? (lb + r.la) * 0.5 : fmax(cb, r.a);
  }
  return r;
}

// The zigzag sums of a block's particles go to an LDS window (three
// components, shaped like the charge window) as int64 fixed
// point at 2^48 per unit, and reach the global FP64 sums once per window
// node.  A segment is summed in the window if its midpoint's offsets from the
// cell are in [-1/2, 3/2] on all axes, as they are for moves of up to two cells
// that stay in the box (a longer one has its relay point at the far cell or face,
// and weights as large as the move; it goes straight to the global sums).  Its
// length is then at most 3 per axis and its weights at most (3/2)^2, so |vv w| <=
// 6.75 < 8 as win_fix needs, and a node's sum of at most kRunMax[1] particles'
// terms (two of 6.75 2^48 each) stays below 2^63; the rounding of each term
// (2^-49) is far below the FP64 summation round-off of the reference's order.
constexpr double kEmFix = 281474976710656.0;          // 2^48

// RESORT as in k_push_dep64.  Bound by latency and instruction issue (VALU about
// 40%, LDS bank conflicts 29% of the CUs' cycles and 81% of the LDS's active ones,
// HBM 3 TB/s); four waves per SIMD (125 VGPRs, 128 with RESORT).  On the
// 18.5M-particle two-stream (128 x 64 x 64), 1.42 ms before: one sum per node
// for a particle that stays in its cell, the flush without divisions and the
// short fixed-point conversion 1.12; four waves instead of three 1.02; the
// windows from the run table instead of a scalar loop per block 0.83, patches
// instead of rows 0.78.  With staged fields (as k_push_dep64) 0.91: the LDS is
// the busier side here.
template <bool RESORT>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4)))
void k_push_em64(State64 s, SpeciesTab sp,
                                                      const double *__restrict__ node, Grid g,
                                                      int ustep, double *__restrict__ jacc,
                                                      int64_t ncell, const Run *__restrict__ runs,
                                                      int *flag, SortDest dst) {
  extern __shared__ __align__(16) unsigned long long win[];
  int is;
  int64_t beg, end;
  Win W, F;
  if (!block_run(s, sp, runs, kRunRow[1], g, kWinRow[1], is, beg, end, W, F)) return;  // uniform
  const int64_t off = sp.off[is];
  const int64_t key0 = (int64_t)is * dst.nkey;
  const int64_t base = RESORT ? off - dst.start[key0] : 0;
  const int wn = W.wx * W.wy * W.wz;  // nodes per component
  zero_win(win, 3 * wn);
  __syncthreads();
  double gustep = (double)ustep;
  double rustep = 1.0 / gustep;
  double qmp = sp.qm[is] * gustep * 0.5;
  double *jx = jacc + ((int64_t)is * 3 + 0) * ncell;
  double *jy = jacc + ((int64_t)is * 3 + 1) * ncell;
  double *jz = jacc + ((int64_t)is * 3 + 2) * ncell;
  for (int64_t mm = beg + threadIdx.x; mm < end; mm += kBlock) {
    const int64_t m = off + mm;
    double x = s.x[m], y = s.y[m], z = s.z[m];
    double vx = s.vx[m], vy = s.vy[m], vz = s.vz[m];
    int64_t d = m;
    int32_t pid = 0;
    if (RESORT) {
      pid = s.pid[m];
      d = base + dst.start[key0 + sort_key_xyz(x, y, z, g, true)] + dst.rank[m];
    }
    domain_guard(x, y, z, g, flag);
    double xlb = x, ylb = y, zlb = z;
    int ib = (int)floor(xlb), jb = (int)floor(ylb), kb = (int)floor(zlb);  // :170-172
    double xb = ib, yb = jb, zb = kb;
    Cic w = cic(xlb, ylb, zlb, ib, jb, kb);
    double f[6];
    gather6<false>(node, g, w, f);
    boris64(vx, vy, vz, f, qmp);
    double xmove = vx * gustep, ymove = vy * gustep, zmove = vz * gustep;
    x = x + xmove;
    y = y + ymove;
    z = z + zmove;
    bool inside = !(x < 0.0 || x >= g.slx || y < 0.0 || y >= g.sly || z < 0.0 || z >= g.slz);
    double px, py, pz;
    Relay rx = relay_axis(x, xlb, xb, ib, g.nx, g.slx, inside, px);
    Relay ry = relay_axis(y, ylb, yb, jb, g.ny, g.sly, inside, py);
    Relay rz = relay_axis(z, zlb, zb, kb, g.nz, g.slz, inside, pz);
    if (!(px >= 0.0 && px <= g.slx && py >= 0.0 && py <= g.sly && pz >= 0.0 && pz <= g.slz))
      atomicOr(flag, kFlagFar);
    const State64 &o = RESORT ? dst.t : s;
    o.x[d] = px;
    o.y[d] = py;
    o.z[d] = pz;
    o.vx[d] = vx;
    o.vy[d] = vy;
    o.vz[d] = vz;
    if (RESORT) o.pid[d] = pid;
    // :717-757
    double xd1 = (rx.r + xlb) * 0.5 - xb, yd1 = (ry.r + ylb) * 0.5 - yb, zd1 = (rz.r + zlb) * 0.5 - zb;
    double vvx1 = (rx.r - xlb) * rustep, vvy1 = (ry.r - ylb) * rustep, vvz1 = (rz.r - zlb) * rustep;
    double vx1w4 = yd1 * zd1, vx1w2 = yd1 - vx1w4, vx1w3 = zd1 - vx1w4, vx1w1 = 1.0 - yd1 - vx1w3;
    double vy1w4 = xd1 * zd1, vy1w2 = xd1 - vy1w4, vy1w3 = zd1 - vy1w4, vy1w1 = 1.0 - xd1 - vy1w3;
    double vz1w4 = xd1 * yd1, vz1w2 = xd1 - vz1w4, vz1w3 = yd1 - vz1w4, vz1w1 = 1.0 - xd1 - vz1w3;
    double xd2 = (rx.la + rx.r) * 0.5 - rx.a, yd2 = (ry.la + ry.r) * 0.5 - ry.a,
           zd2 = (rz.la + rz.r) * 0.5 - rz.a;
    double vvx2 = (rx.la - rx.r) * rustep, vvy2 = (ry.la - ry.r) * rustep,
           vvz2 = (rz.la - rz.r) * rustep;
    double vx2w4 = yd2 * zd2, vx2w2 = yd2 - vx2w4, vx2w3 = zd2 - vx2w4, vx2w1 = 1.0 - yd2 - vx2w3;
    double vy2w4 = xd2 * zd2, vy2w2 = xd2 - vy2w4, vy2w3 = zd2 - vy2w4, vy2w1 = 1.0 - xd2 - vy2w3;
    double vz2w4 = xd2 * yd2, vz2w2 = xd2 - vz2w4, vz2w3 = yd2 - vz2w4, vz2w1 = 1.0 - xd2 - vz2w3;
    const double ax1[4] = {vx1w1, vx1w2, vx1w3, vx1w4}, ay1[4] = {vy1w1, vy1w2, vy1w3, vy1w4},
                 az1[4] = {vz1w1, vz1w2, vz1w3, vz1w4};
    const double ax2[4] = {vx2w1, vx2w2, vx2w3, vx2w4}, ay2[4] = {vy2w1, vy2w2, vy2w3, vy2w4},
                 az2[4] = {vz2w1, vz2w2, vz2w3, vz2w4};
    // the 12 contributions of a segment (:759-789), in the window when its cell
    // and the next node along every axis are inside; value(c, k) is component
    // c's contribution with its weight k
    auto seg = [&](int i, int j, int k, bool fits, auto value) {
      const int li = wrapn(i - W.ox, g.nx), lj = wrapn(j - W.oy, g.ny), lk = wrapn(k - W.oz, g.nz);
      int li1, lj1, lk1;
      if (fits && li < W.wx && lj < W.wy && lk < W.wz && win_next(li, W.wx, g.nx, li1) &&
          win_next(lj, W.wy, g.ny, lj1) && win_next(lk, W.wz, g.nz, lk1)) {
        const int dx = li1 - li, dy = (lj1 - lj) * W.wx, dz = (lk1 - lk) * (W.wx * W.wy);
        unsigned long long *p = win + (lk * W.wy + lj) * W.wx + li;
        atomicAdd(p, win_fix(value(0, 0)));
        atomicAdd(p + dy, win_fix(value(0, 1)));
        atomicAdd(p + dz, win_fix(value(0, 2)));
        atomicAdd(p + dy + dz, win_fix(value(0, 3)));
        p += wn;
        atomicAdd(p, win_fix(value(1, 0)));
        atomicAdd(p + dx, win_fix(value(1, 1)));
        atomicAdd(p + dz, win_fix(value(1, 2)));
        atomicAdd(p + dx + dz, win_fix(value(1, 3)));
        p += wn;
        atomicAdd(p, win_fix(value(2, 0)));
        atomicAdd(p + dx, win_fix(value(2, 1)));
        atomicAdd(p + dy, win_fix(value(2, 2)));
        atomicAdd(p + dx + dy, win_fix(value(2, 3)));
      } else {
        const int i1 = i + 1, j1 = j + 1, k1 = k + 1;
        atomicAdd(jx + cidx(g, i, j, k), value(0, 0));
        atomicAdd(jx + cidx(g, i, j1, k), value(0, 1));
        atomicAdd(jx + cidx(g, i, j, k1), value(0, 2));
        atomicAdd(jx + cidx(g, i, j1, k1), value(0, 3));
        atomicAdd(jy + cidx(g, i, j, k), value(1, 0));
        atomicAdd(jy + cidx(g, i1, j, k), value(1, 1));
        atomicAdd(jy + cidx(g, i, j, k1), value(1, 2));
        atomicAdd(jy + cidx(g, i1, j, k1), value(1, 3));
        atomicAdd(jz + cidx(g, i, j, k), value(2, 0));
        atomicAdd(jz + cidx(g, i1, j, k), value(2, 1));
        atomicAdd(jz + cidx(g, i, j1, k), value(2, 2));
        atomicAdd(jz + cidx(g, i1, j1, k), value(2, 3));
      }
    };
    auto near = [](double a, double b, double c) {
      return fabs(a - 0.5) <= 1.0 && fabs(b - 0.5) <= 1.0 && fabs(c - 0.5) <= 1.0;
    };
    const bool near2 = near(xd2, yd2, zd2);
    // a particle that stays in its cell has both segments there: one sum (of a
    // move within the cell, or beyond the face from a position of exactly L) per
    // node, the second segment's own sums only for the particles that changed cell
    const bool same = rx.ia == ib && ry.ia == jb && rz.ia == kb;
    const double sx2 = same ? vvx2 : 0.0, sy2 = same ? vvy2 : 0.0, sz2 = same ? vvz2 : 0.0;
    seg(ib, jb, kb, near(xd1, yd1, zd1) && (!same || near2), [&](int c, int k) {
      return c == 0 ? vvx1 * ax1[k] + sx2 * ax2[k]
                    : (c == 1 ? vvy1 * ay1[k] + sy2 * ay2[k] : vvz1 * az1[k] + sz2 * az2[k]);
    });
    if (!same)
      seg(rx.ia, ry.ia, rz.ia, near2, [&](int c, int k) {
        return c == 0 ? vvx2 * ax2[k] : (c == 1 ? vvy2 * ay2[k] : vvz2 * az2[k]);
      });
  }
  __syncthreads();
  double *const acc[3] = {jx, jy, jz};
  flush_win<3>(win, W, acc, g, 1.0 / kEmFix);
}

dim3 species_grid(const SpeciesTab &sp) {
  int64_t mx = 1;
  for (int s = 0; s < sp.nspec; s++) mx = sp.cnt[s] > mx ? sp.cnt[s] : mx;
  return dim3((unsigned)((mx + kBlock - 1) / kBlock), (unsigned)sp.nspec, 1);
}


// A block's sums for the face slots that its particles reach, in LDS: open
// addressing, at most kProbe tries, the rest goes to the global array.  The
// face nodes collect one particle in twenty (64^3 cells), neighbours in the
// state on the same few nodes: one global atomic per block and node instead of
// four per particle.
template <class V, int kSlots>
struct FaceTable {
  static constexpr int kProbe = 8;
  unsigned long long key[kSlots];
  V sum[kSlots];
  __device__ __forceinline__ void clear() {
    for (int h = threadIdx.x; h < kSlots; h += blockDim.x) {
      key[h] = ~0ull;
      sum[h] = 0;
    }
  }
  __device__ __forceinline__ void add(V *face, int64_t slot, V v) {
    const unsigned long long want = (unsigned long long)slot;
    static_assert(kSlots == 1 || kSlots == 1 << 10, "hash");
    int h = (int)(((uint32_t)want * 2654435769u) >> 22);
    for (int t = 0; t < kProbe; t++) {
      unsigned long long k = key[h];
      if (k == ~0ull) k = atomicCAS(&key[h], ~0ull, want);
      if (k == ~0ull || k == want) {
        atomicAdd(&sum[h], v);
        return;
      }
      h = (h + 1) & (kSlots - 1);
    }
    atomicAdd(face + slot, v);
  }
  __device__ __forceinline__ void flush(V *face) {
    for (int h = threadIdx.x; h < kSlots; h += blockDim.x)
      if (key[h] != ~0ull) atomicAdd(face + key[h], sum[h]);
  }
};

// The weights that the reference's charge puts on nodes with index n on some
// axis (charge.F90:152-210 with int(): a particle in cell n - 1, or at a
// position of exactly L, reaches them), kept per species in the upper-face
// arrays.  A weight on node n + 1 (only a position of exactly L has one, of
// size zero) is dropped, as the reference's border exchange overwrites that
// node.
// Streams the positions (24 bytes per particle).  TABLE, for a state in order: a
// block's kFacePart particles sum what they add in LDS first.  8.4M particles on
// 64^3 cells, sorted: 148 us with an atomic per weight, 59 with the table; in no
// order the table gathers little (25 us more on 4 to 8M particles).
constexpr int kFacePer = 4, kFacePart = kFacePer * kBlock;
template <bool TABLE>
__global__ __launch_bounds__(kBlock) void k_faces64(State64 s, SpeciesTab sp, Grid g,
                                                    double *__restrict__ face, int64_t nf) {
  __shared__ FaceTable<double, TABLE ? 1024 : 1> tab;
  const int is = blockIdx.y;
  const int64_t m0 = (int64_t)blockIdx.x * kFacePart;
  if (m0 >= sp.cnt[is]) return;  // uniform
  double px[kFacePer], py[kFacePer], pz[kFacePer];
  bool on[kFacePer], any = false;
#pragma unroll
  for (int u = 0; u < kFacePer; u++) {
    int64_t m = m0 + u * kBlock + threadIdx.x;
    on[u] = m < sp.cnt[is];
    m = sp.off[is] + (on[u] ? m : m0);
    px[u] = s.x[m];
    py[u] = s.y[m];
    pz[u] = s.z[m];
  }
#pragma unroll
  for (int u = 0; u < kFacePer; u++) {
    double &x = px[u], &y = py[u], &z = pz[u];
    x = x >= 0.0 ? (x <= g.slx ? x : g.slx) : 0.0;
    y = y >= 0.0 ? (y <= g.sly ? y : g.sly) : 0.0;
    z = z >= 0.0 ? (z <= g.slz ? z : g.slz) : 0.0;
    on[u] = on[u] && ((int)x >= g.nx - 1 || (int)y >= g.ny - 1 || (int)z >= g.nz - 1);
    any = any || on[u];
  }
  if (TABLE) {
    if (!__syncthreads_or(any)) return;
    tab.clear();
    __syncthreads();
  }
  const double qc = sp.q[is];
  double *f = face + (int64_t)is * nf;
#pragma unroll
  for (int u = 0; u < kFacePer; u++) {
    if (!on[u]) continue;
    const double x = px[u], y = py[u], z = pz[u];
    const int i = (int)x, j = (int)y, k = (int)z;
    const Cic w = cic(x, y, z, i, j, k);
    const int ci[8] = {i, i + 1, i + 1, i, i, i + 1, i + 1, i};
    const int cj[8] = {j, j, j + 1, j + 1, j, j, j + 1, j + 1};
    const int ck[8] = {k + 1, k + 1, k + 1, k + 1, k, k, k, k};
    const double v[8] = {w.v1, w.v2, w.v3, w.v4, w.v5, w.v6, w.v7, w.v8};
#pragma unroll
    for (int q = 0; q < 8; q++) {
      if (ci[q] > g.nx || cj[q] > g.ny || ck[q] > g.nz) continue;
      const int64_t fi = face_index(g, ci[q], cj[q], ck[q]);
      if (fi < 0) continue;
      if (TABLE) tab.add(f, fi, v[q] * qc);
      else atomicAdd(f + fi, v[q] * qc);
    }
  }
  if (TABLE) {
    __syncthreads();
    tab.flush(f);
  }
}

}  // namespace

void launch_relocate64(emg_ctx *c) {
  int64_t nn = (int64_t)(c->g.nx + 1) * (c->g.ny + 1) * (c->g.nz + 1);
  const emg_config &f = c->cfg;
  timer_begin(c, kTRelocate);
  hipLaunchKernelGGL(k_relocate, dim3((unsigned)((nn + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, eb_view(c),
                     c->cfg.precision == EMG_PLAIN_FP64 ? c->node64 : nullptr,
                     c->cfg.precision == EMG_FP32_FIXED ? c->node32 : nullptr, c->ncell, f.e0[0],
                     f.e0[1], f.e0[2], f.b0[0], f.b0[1], f.b0[2]);
  timer_end(c, kTRelocate);
  if (!capturing(c)) c->nodes_b_valid = true;  // (recorded, not done)
}

void launch_positn64(emg_ctx *c, int ustep) {
  timer_begin(c, kTPush);
  hipLaunchKernelGGL(k_positn64, species_grid(c->sp), dim3(kBlock), 0, c->stream, c->s64, c->sp,
                     c->g, ustep, c->dflag);
  timer_end(c, kTPush);
}

// The grid of a kernel of table `which`: the last sort's run table when it is
// there (one block per run), else (slices, species) with runs = nullptr; and
// its LDS: `comps` windows of the runs' shape, and (patched, fields) the staged
// field nodes.
static dim3 block_grid(const emg_ctx *c, int which, int comps, bool fields, const Run *&runs,
                       size_t &lds, bool &patched) {
  const bool table = c->runs_valid && c->nruns[which] > 0;
  patched = table && c->sort_patched;
  lds = sizeof(unsigned long long) * comps * (patched ? kWinPatch[which] : kWinRow[which].cap);
  if (patched && fields) lds += sizeof(double2) * 3 * kFieldCap;
  if (table) {
    runs = c->runs[which];
    return dim3((unsigned)c->nruns[which]);
  }
  runs = nullptr;
  int64_t mx = 1;
  for (int q = 0; q < c->sp.nspec; q++) mx = c->sp.cnt[q] > mx ? c->sp.cnt[q] : mx;
  return dim3((unsigned)((mx + kRunRow[which] - 1) / kRunRow[which]), c->sp.nspec);
}

// An unsorted state of at least this many particles is worth binning (five
// launches more; eight atomics per particle fewer).
constexpr int64_t kTileMin = 1 << 17;

// whether the charge of the state goes through the tiles: in no order, and the
// workspace can be had (it cannot be allocated while the stream is captured)
static bool tiles64(emg_ctx *c) {
  int64_t total = 0;
  for (int s = 0; s < c->sp.nspec; s++) total += c->sp.cnt[s];
  if (c->runs_valid || c->ordered || total < kTileMin) return false;
  return c->bins.rec || (!capturing(c) && bins_alloc(c) == EMG_OK);
}

static void launch_tiles64(emg_ctx *c) {
  const BinTiles at = bin_tiles(c->g);
  const size_t lds = sizeof(double) * kTileNodes * c->sp.nspec;
  int64_t done[EMG_MAX_SPECIES] = {};
  while (const int64_t total = bin_pass(c, done)) {
    // as the adjoint step: 512 workgroups or more, of 16 rounds at least
    int64_t split = (512 + at.n - 1) / at.n;
    split = std::min<int64_t>(split, total / ((int64_t)at.n * kTileBlock * 16) + 1);
    hipLaunchKernelGGL(k_tile_charge, dim3(at.n, (unsigned)split), dim3(kTileBlock), lds, c->stream,
                       c->bins.rec, c->bins.start, at, c->sp, c->g, c->rho64, c->ncell, c->dflag);
  }
}

void launch_push_es64(emg_ctx *c, int ustep, bool resort) {
  launch_zero(c->rho64, sizeof(double) * c->ncell * c->sp.nspec, c->stream);
  timer_begin(c, kTPush);
  const Run *runs;
  size_t lds;
  bool patched;
  const dim3 grid = block_grid(c, 0, 1, true, runs, lds, patched);
  const SortDest dst = resort ? sort64_dest(c) : SortDest{};
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, c->stream, c->s64, c->sp, c->node64, c->g,
                       ustep, c->rho64, c->ncell, runs, c->dflag, dst);
  };
  if (tiles64(c)) {
    go(k_push_dep64<false, false, false>);
    launch_tiles64(c);
  } else if (patched) {
    resort ? go(k_push_dep64<true, true>) : go(k_push_dep64<false, true>);
  } else {
    resort ? go(k_push_dep64<true, false>) : go(k_push_dep64<false, false>);
  }
  timer_end(c, kTPush);
}

void launch_deposit64(emg_ctx *c) {
  launch_zero(c->rho64, sizeof(double) * c->ncell * c->sp.nspec, c->stream);
  timer_begin(c, kTDeposit);
  if (tiles64(c)) {
    launch_tiles64(c);
    timer_end(c, kTDeposit);
    return;
  }
  const Run *runs;
  size_t lds;
  bool patched;
  const dim3 grid = block_grid(c, 0, 1, false, runs, lds, patched);
  hipLaunchKernelGGL(k_deposit64, grid, dim3(kBlock), lds, c->stream, c->s64, c->sp, c->g, c->rho64,
                     c->ncell, runs, c->dflag);
  timer_end(c, kTDeposit);
}

void launch_push_em64(emg_ctx *c, int ustep, bool resort) {
  launch_zero(c->j64, sizeof(double) * 3 * c->ncell * c->sp.nspec, c->stream);
  timer_begin(c, kTPush);
  const Run *runs;
  size_t lds;
  bool patched;
  const dim3 grid = block_grid(c, 1, 3, false, runs, lds, patched);
  const SortDest dst = resort ? sort64_dest(c) : SortDest{};
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kBlock), lds, c->stream, c->s64, c->sp, c->node64, c->g,
                       ustep, c->j64, c->ncell, runs, c->dflag, dst);
  };
  resort ? go(k_push_em64<true>) : go(k_push_em64<false>);
  timer_end(c, kTPush);
}

void launch_faces64(emg_ctx *c) {
  const int64_t nf = face_len(c->g);
  launch_zero(c->face, sizeof(double) * nf * c->sp.nspec, c->stream);
  int64_t mx = 1;
  for (int q = 0; q < c->sp.nspec; q++) mx = c->sp.cnt[q] > mx ? c->sp.cnt[q] : mx;
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)((mx + kFacePart - 1) / kFacePart), c->sp.nspec),
                       dim3(kBlock), 0, c->stream, c->s64, c->sp, c->g, (double *)c->face, nf);
  };
  c->runs_valid || c->ordered ? go(k_faces64<true>) : go(k_faces64<false>);
}

}  // namespace emg
