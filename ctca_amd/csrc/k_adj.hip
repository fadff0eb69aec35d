// k_adj.hip -- reverse (adjoint) step of the FP64 electrostatic push, for the
// differentiable window of the torch harness.
//
// Forward step k (emg_push_es in EMG_PLAIN_FP64, psolve2.F90:137-318) maps
// (x_k, v_k) to
//   a      = qmp * E(x_k)                      (trilinear gather of nodal E)
//   v_k+1  = M (v_k + a) + a                   (Boris; M the rotation by b = qmp B)
//   x_k+1  = x_k + ustep * v_k+1               (periodic wrap: a translation)
// With lambda_x, lambda_v the adjoints of (x_k+1, v_k+1), the adjoints of
// (x_k, v_k) are
//   w        = lambda_v + ustep * lambda_x
//   lambda_a = M^T w + w,   lambda_v <- M^T w  (M^T is the rotation by -b)
//   lambda_x <- lambda_x + sum_c lambda_a_c * qmp * grad E_c(x_k)
// and qmp * lambda_a is scattered with the same trilinear weights onto a
// nodal adjoint field (the transpose of the gather, binned by tiles: below),
// from which the host
// forms the adjoint of rho through the field solve; the contribution of
// x_k to rho is then added by k_adj_density: lambda_x += q * grad g(x_k).
// B enters as a constant (the electrostatic path keeps B static; the
// gradient of a non-uniform B is not part of the step adjoint).
#include <algorithm>

#include "emg_internal.h"

namespace emg {
namespace {

__device__ __forceinline__ int64_t nodal(const Grid &g, int i, int j, int k) {
  return ((int64_t)k * (g.ny + 1) + j) * (g.nx + 1) + i;
}

__device__ __forceinline__ int64_t periodic(const Grid &g, int i, int j, int k) {
  return ((int64_t)(k == g.nz ? 0 : k) * g.ny + (j == g.ny ? 0 : j)) * g.nx + (i == g.nx ? 0 : i);
}

struct Tri {
  int i, j, k;
  double wx[2], wy[2], wz[2];
};

// cell and weights of the reference's trilinear interpolation (int() cells,
// psolve2.F90:154-183), positions in [0, L]; the cell is held in the grid for one
// beyond, which a push that reported it as moved too far may have left
__device__ __forceinline__ Tri tri(double x, double y, double z, const Grid &g) {
  Tri t;
  t.i = min(max((int)x, 0), g.nx - 1);
  t.j = min(max((int)y, 0), g.ny - 1);
  t.k = min(max((int)z, 0), g.nz - 1);
  double x1 = x - t.i, y1 = y - t.j, z1 = z - t.k;
  t.wx[0] = 1.0 - x1;
  t.wx[1] = x1;
  t.wy[0] = 1.0 - y1;
  t.wy[1] = y1;
  t.wz[0] = 1.0 - z1;
  t.wz[1] = z1;
  return t;
}

// gradient of the trilinear interpolant of corner values s[c] (c = a + 2b + 4c')
__device__ __forceinline__ void tri_grad(const Tri &t, const double s[8], double gr[3]) {
  gr[0] = gr[1] = gr[2] = 0.0;
#pragma unroll
  for (int q = 0; q < 8; q++) {
    int a = q & 1, b = (q >> 1) & 1, c = q >> 2;
    double sx = a ? 1.0 : -1.0, sy = b ? 1.0 : -1.0, sz = c ? 1.0 : -1.0;
    gr[0] += s[q] * sx * t.wy[b] * t.wz[c];
    gr[1] += s[q] * t.wx[a] * sy * t.wz[c];
    gr[2] += s[q] * t.wx[a] * t.wy[b] * sz;
  }
}

// rotation u -> u + bor ((u + u x b) x b) of the Boris push; with -b it is
// the transpose of the rotation with b
__device__ __forceinline__ void rotate(double u[3], const double b[3]) {
  double bor = 2.0 / (1.0 + b[0] * b[0] + b[1] * b[1] + b[2] * b[2]);
  double tx = u[0] + u[1] * b[2] - u[2] * b[1];
  double ty = u[1] + u[2] * b[0] - u[0] * b[2];
  double tz = u[2] + u[0] * b[1] - u[1] * b[0];
  u[0] += bor * (ty * b[2] - tz * b[1]);
  u[1] += bor * (tz * b[0] - tx * b[2]);
  u[2] += bor * (tx * b[1] - ty * b[0]);
}

// The particles of a window are in no spatial order (their order is that of
// every saved state).  Stepped in that order, the kernel gathered 24 x 16 bytes
// from random cells and sent one global FP64 atomic per particle, node and
// component, at 22 G atomics/s: 9.28 ms for 8.8M particles on 64^3 cells, whose
// state is 0.2 ms of traffic.  So a step bins the particles by tiles first
// (k_bin.hip), and k_adj_step64 takes one workgroup per tile: its nodes' E and B
// staged in LDS, the reverse step of its particles (their adjoints are 64-byte
// records, so an access at a random particle is one line), the transposed
// gather summed in an LDS tile of FP64 nodes, each of which reaches memory once.
// At the same size: 0.08 (count) + 0.26 (bin) + 0.50 ms, bound by the random
// 64-byte lines of the adjoints.  (Binning only the scatter, with the gather in
// slot order, took 0.08 + 2.22 + 0.18 ms.)
constexpr int kAdjBlock = 512;

// The reverse step of tile blockIdx.x's records (slice blockIdx.y of
// gridDim.y).  A node strictly inside the tile belongs to this tile alone:
// with one workgroup per tile it is added to adj_e without an atomic.
__global__ __launch_bounds__(kAdjBlock) void k_adj_step64(double *__restrict__ lam, SpeciesTab sp,
                                                         const double *__restrict__ node, Grid g,
                                                         int ustep,
                                                         const BinRec *__restrict__ rec,
                                                         const int64_t *__restrict__ start,
                                                         BinTiles at,
                                                         double *__restrict__ adj_e) {
  constexpr int N = kBinTile + 1, NN = N * N * N;
  __shared__ double2 fs[3 * NN];  // E and B of the tile's nodes
  __shared__ double acc[3 * NN];
  const int tl = blockIdx.x;
  const int64_t beg = start[tl], end = start[tl + 1];
  const int64_t step = (int64_t)gridDim.y * kAdjBlock;
  if (beg + (int64_t)blockIdx.y * kAdjBlock >= end) return;  // uniform over the block
  const int ox = (tl % at.ntx) * kBinTile, oy = (tl / at.ntx) % at.nty * kBinTile,
            oz = tl / (at.ntx * at.nty) * kBinTile;
  const int tx = min(kBinTile, g.nx - ox), ty = min(kBinTile, g.ny - oy),
            tz = min(kBinTile, g.nz - oz);
  for (int q = threadIdx.x; q < 3 * NN; q += kAdjBlock) {
    acc[q] = 0.0;
    const int nq = q / 3, c = q - 3 * nq;
    const int i = nq % N, j = (nq / N) % N, k = nq / (N * N);
    if (i <= tx && j <= ty && k <= tz)
      fs[q] = reinterpret_cast<const double2 *>(node + 8 * nodal(g, ox + i, oy + j, oz + k))[c];
  }
  __syncthreads();
  const double gustep = (double)ustep;
  int64_t m = beg + (int64_t)blockIdx.y * kAdjBlock + threadIdx.x;
  double2 r0{}, r1{};
  if (m < end) {
    r0 = reinterpret_cast<const double2 *>(rec + m)[0];
    r1 = reinterpret_cast<const double2 *>(rec + m)[1];
  }
  for (; m < end; m += step) {
    const Tri t = tri(r0.x, r0.y, r1.x, g);
    const int64_t ms = __double_as_longlong(r1.y);
    double2 *lp = reinterpret_cast<double2 *>(lam + 8 * (ms & 0x00ffffffffffffffll));
    const double2 l0 = lp[0], l1 = lp[1], l2 = lp[2];
    if (m + step < end) {  // the next record, while this one's adjoints arrive
      r0 = reinterpret_cast<const double2 *>(rec + m + step)[0];
      r1 = reinterpret_cast<const double2 *>(rec + m + step)[1];
    }
    const double qmp = sp.qm[ms >> 56] * gustep * 0.5;
    const int nc = ((t.k - oz) * N + (t.j - oy)) * N + (t.i - ox);
    double bf[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int a = q & 1, b = (q >> 1) & 1, c = q >> 2;
      const double2 *f = fs + 3 * (nc + (c * N + b) * N + a);
      const double w = t.wx[a] * t.wy[b] * t.wz[c];
      bf[0] += w * f[1].y;
      bf[1] += w * f[2].x;
      bf[2] += w * f[2].y;
    }
    double nb[3] = {-bf[0] * qmp, -bf[1] * qmp, -bf[2] * qmp};
    const double w3[3] = {l1.y + gustep * l0.x, l2.x + gustep * l0.y, l2.y + gustep * l1.x};
    double mt[3] = {w3[0], w3[1], w3[2]};
    rotate(mt, nb);
    const double la[3] = {mt[0] + w3[0], mt[1] + w3[1], mt[2] + w3[2]};
    // lambda_x += qmp * grad (lambda_a . E)(x_k), and qmp * lambda_a onto the nodes
    double sdot[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int a = q & 1, b = (q >> 1) & 1, c = q >> 2;
      const int nq = nc + (c * N + b) * N + a;
      const double2 *f = fs + 3 * nq;
      sdot[q] = la[0] * f[0].x + la[1] * f[0].y + la[2] * f[1].x;
      const double w = qmp * t.wx[a] * t.wy[b] * t.wz[c];
      atomicAdd(&acc[nq], w * la[0]);
      atomicAdd(&acc[nq + NN], w * la[1]);
      atomicAdd(&acc[nq + 2 * NN], w * la[2]);
    }
    double gr[3];
    tri_grad(t, sdot, gr);
    lp[0] = make_double2(l0.x + qmp * gr[0], l0.y + qmp * gr[1]);
    lp[1] = make_double2(l1.x + qmp * gr[2], mt[0]);
    lp[2] = make_double2(mt[1], mt[2]);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < NN; q += kAdjBlock) {
    const int i = q % N, j = (q / N) % N, k = q / (N * N);
    if (i > tx || j > ty || k > tz) continue;
    double *d = adj_e + 3 * periodic(g, ox + i, oy + j, oz + k);
    const bool own = gridDim.y == 1 && i > 0 && i < tx && j > 0 && j < ty && k > 0 && k < tz;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const double v = acc[c * NN + q];
      if (own) d[c] += v;
      else if (v != 0.0) atomicAdd(d + c, v);
    }
  }
}

struct SpeciesFactors {
  double v[EMG_MAX_SPECIES];
};

// lambda_x += qfac[is] * grad g(x) for the trilinear interpolant of the
// periodic nodal scalar g (the adjoint of the particle's CIC charge)
__global__ __launch_bounds__(kBlock) void k_adj_density64(State64 s, double *__restrict__ lam, SpeciesTab sp,
                                                         Grid g, const double *__restrict__ gn, SpeciesFactors qfac) {
  int is = blockIdx.y;
  double f = qfac.v[is];
  if (f == 0.0) return;
  int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= sp.cnt[is]) return;
  m += sp.off[is];
  double *l = lam + 8 * m;
  const double2 l0 = *reinterpret_cast<const double2 *>(l);
  const double lz = l[2];
  Tri t = tri(s.x[m], s.y[m], s.z[m], g);
  // the two nodes of each x edge in one 16-byte load (8-byte aligned); in the
  // last cell the second one is node 0 of the row
  double v[8];
  const int i0 = min(t.i, g.nx - 2);
  const bool last = t.i != i0;
  const int j1 = t.j + 1 == g.ny ? 0 : t.j + 1, k1 = t.k + 1 == g.nz ? 0 : t.k + 1;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const double *row = gn + ((int64_t)(q >> 1 ? k1 : t.k) * g.ny + (q & 1 ? j1 : t.j)) * g.nx;
    __builtin_memcpy(&v[2 * q], row + i0, 2 * sizeof(double));
    if (last) {
      v[2 * q] = v[2 * q + 1];
      v[2 * q + 1] = row[0];
    }
  }
  double gr[3];
  tri_grad(t, v, gr);
  *reinterpret_cast<double2 *>(l) = make_double2(l0.x + f * gr[0], l0.y + f * gr[1]);
  l[2] = lz + f * gr[2];
}

// per-species sums of lambda_v: kVsumBlocks block partials per species, then
// one block adds them in block order: 0.11 ms at 8.8M particles.  (Three atomics
// per block of 256 particles, on six addresses, took 0.79.)
constexpr int kVsumBlocks = 512;

__device__ __forceinline__ void vsum_block(double v[3], double *out) {
  __shared__ double red[3][kBlock];
  for (int d = 0; d < 3; d++) red[d][threadIdx.x] = v[d];
  __syncthreads();
  for (int o = kBlock / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o)
      for (int d = 0; d < 3; d++) red[d][threadIdx.x] += red[d][threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x < 3) out[threadIdx.x] = red[threadIdx.x][0];
}

__global__ __launch_bounds__(kBlock) void k_adj_vsum(const double *__restrict__ lam, SpeciesTab sp,
                                                    double *part) {
  const int is = blockIdx.y;
  double v[3] = {0.0, 0.0, 0.0};
  for (int64_t m = (int64_t)blockIdx.x * kBlock + threadIdx.x; m < sp.cnt[is];
       m += (int64_t)kVsumBlocks * kBlock) {
    const double *l = lam + 8 * (sp.off[is] + m);
    v[0] += l[3];
    v[1] += l[4];
    v[2] += l[5];
  }
  vsum_block(v, part + 3 * ((int64_t)is * kVsumBlocks + blockIdx.x));
}

__global__ __launch_bounds__(kBlock) void k_adj_vsum_final(const double *part, double *out,
                                                          const int *dflag, int *hflag) {
  const int is = blockIdx.x;
  if (is == 0 && threadIdx.x == 0) *hflag = *dflag;
  double v[3] = {0.0, 0.0, 0.0};
  for (int k = threadIdx.x; k < kVsumBlocks; k += kBlock)
    for (int d = 0; d < 3; d++) v[d] += part[3 * ((int64_t)is * kVsumBlocks + k) + d];
  vsum_block(v, out + 3 * is);
}

dim3 species_blocks(const SpeciesTab &sp) {
  int64_t mx = 1;
  for (int s = 0; s < sp.nspec; s++) mx = sp.cnt[s] > mx ? sp.cnt[s] : mx;
  return dim3((unsigned)((mx + kBlock - 1) / kBlock), sp.nspec);
}

}  // namespace

void launch_adj_step64(emg_ctx *c, int ustep) {
  launch_zero(c->adj_e, sizeof(double) * 3 * c->ncell, c->stream);
  const BinTiles at = bin_tiles(c->g);
  int64_t done[EMG_MAX_SPECIES] = {};
  while (const int64_t total = bin_pass(c, done)) {
    // about 512 workgroups or more (two per CU), of 16 rounds of records at least
    int64_t split = (512 + at.n - 1) / at.n;
    split = std::min<int64_t>(split, total / ((int64_t)at.n * kAdjBlock * 16) + 1);
    hipLaunchKernelGGL(k_adj_step64, dim3(at.n, (unsigned)split), dim3(kAdjBlock), 0, c->stream,
                       c->lam, c->sp, c->node64, c->g, ustep, c->bins.rec, c->bins.start, at,
                       c->adj_e);
  }
}

void launch_adj_density64(emg_ctx *c, const double *qfac) {
  SpeciesFactors f{};
  for (int s = 0; s < c->sp.nspec; s++) f.v[s] = qfac[s];
  hipLaunchKernelGGL(k_adj_density64, species_blocks(c->sp), dim3(kBlock), 0, c->stream, c->s64,
                     c->lam, c->sp, c->g, c->adj_g, f);
}

void launch_adj_vsum(emg_ctx *c, double *part, double *out) {
  hipLaunchKernelGGL(k_adj_vsum, dim3(kVsumBlocks, c->sp.nspec), dim3(kBlock), 0, c->stream, c->lam,
                     c->sp, part);
  hipLaunchKernelGGL(k_adj_vsum_final, dim3(c->sp.nspec), dim3(kBlock), 0, c->stream, part, out,
                     c->dflag, c->hflag);
}

int64_t adj_vsum_need() { return (int64_t)3 * EMG_MAX_SPECIES * kVsumBlocks; }

}  // namespace emg
