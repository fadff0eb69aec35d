// k_yee.hip -- the EM field update on the device, on the library's copy of
// the staggered Yee array eb(6, lo:hi) (ghosts included; one array per
// component), for one periodic rank:
//   bfield  (bfield.F90:38-52): B += curl-difference of E (a half step);
//   efield  (efield.F90:55-72): E += tcs curl-difference of B - dlt aj, with
//           aj the folded current of the last emg_push_em;
//   energy  (energy.F90:52-70): the field part engeb.
// Every point of the array, ghosts included, is computed from the periodic
// images of its neighbours: a ghost gets exactly the value of its image,
// which is what the reference's border exchange gives it after the update on
// one periodic rank.  The updates read only the other field, so they run in
// place.  They are bound by memory, and every access is a coalesced 8-byte one:
// with the boundary's six-component records (an update rewrites 24 bytes of
// each 48) a B half step took 37 us and an E step 44 us on 131 x 131 x 67
// points, 20 and 32 us now.  Expression order as in the reference; built without FP contraction.
#include "emg_internal.h"

namespace emg {
namespace {

constexpr int BX = 3, BY = 4, BZ = 5;  // eb components: EX EY EZ BX BY BZ

__device__ __forceinline__ bool my_point(const EbView &v, int64_t &o, int &i, int &j, int &k) {
  o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= v.np) return false;
  point_of(o, v.ext[0], v.ext[1], i, j, k);
  i += v.lo[0];
  j += v.lo[1];
  k += v.lo[2];
  return true;
}

// n uploaded records (six components per point) into the component arrays from
// point o0 on
__global__ __launch_bounds__(kBlock) void k_eb_split(const double *__restrict__ rec, EbView v,
                                                     int64_t o0, int64_t n) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= n) return;
  const double2 *r = reinterpret_cast<const double2 *>(rec + 6 * o);
  double2 a[3];
#pragma unroll
  for (int q = 0; q < 3; q++) a[q] = r[q];
#pragma unroll
  for (int q = 0; q < 3; q++) {
    v.eb[(2 * q) * v.np + o0 + o] = a[q].x;
    v.eb[(2 * q + 1) * v.np + o0 + o] = a[q].y;
  }
}

__global__ __launch_bounds__(kBlock) void k_bfield(EbView v) {
  int64_t o;
  int i, j, k;
  if (!my_point(v, o, i, j, k)) return;
  const double *ex = v.eb, *ey = v.eb + v.np, *ez = v.eb + 2 * v.np;
  const int64_t p0 = v.img(i, j, k), pk = v.img(i, j, k + 1), pj = v.img(i, j + 1, k),
                pi = v.img(i + 1, j, k);
  const double x0 = ex[p0], y0 = ey[p0], z0 = ez[p0];
  double *bx = v.eb + BX * v.np + o, *by = v.eb + BY * v.np + o, *bz = v.eb + BZ * v.np + o;
  const double nx = *bx + ey[pk] - y0 - ez[pj] + z0;
  const double ny = *by + ez[pi] - z0 - ex[pk] + x0;
  const double nz = *bz + ex[pj] - x0 - ey[pi] + y0;
  *bx = nx;
  *by = ny;
  *bz = nz;
}

struct CurrentView {
  const void *jacc;  // nspec x 3 x ncell: int64 fixed point (FIX) or FP64 sums
  double q[EMG_MAX_SPECIES];
  int nspec;
  int64_t ncell;
};

// aj(d) of periodic cell c: sum over species of J(is) q(is), in species order,
// each term added with one fused multiply-add (the read-out of
// emg_get_current, so the E update takes exactly the current it reports)
template <bool FIX>
__device__ __forceinline__ double aj_at(const CurrentView &J, int d, int64_t c) {
  double v = 0.0;
  for (int s = 0; s < J.nspec; s++) {
    const int64_t q = ((int64_t)s * 3 + d) * J.ncell + c;
    const double js = FIX ? (double)(long long)((const unsigned long long *)J.jacc)[q] * (1.0 / kJScale)
                          : ((const double *)J.jacc)[q];
    v = fma(js, J.q[s], v);
  }
  return v;
}

template <bool FIX>
__global__ __launch_bounds__(kBlock) void k_efield(EbView v, CurrentView J, double tcs,
                                                   double dlt) {
  int64_t o;
  int i, j, k;
  if (!my_point(v, o, i, j, k)) return;
  const int64_t c = ((int64_t)periodic_index(k, v.g.nz) * v.g.ny + periodic_index(j, v.g.ny)) *
                        v.g.nx +
                    periodic_index(i, v.g.nx);
  const double *bx = v.eb + BX * v.np, *by = v.eb + BY * v.np, *bz = v.eb + BZ * v.np;
  const int64_t p0 = v.img(i, j, k), pj = v.img(i, j - 1, k), pk = v.img(i, j, k - 1),
                pi = v.img(i - 1, j, k);
  const double x0 = bx[p0], y0 = by[p0], z0 = bz[p0];
  double *ex = v.eb + o, *ey = v.eb + v.np + o, *ez = v.eb + 2 * v.np + o;
  const double nx = *ex + tcs * (z0 - bz[pj] - y0 + by[pk]) - dlt * aj_at<FIX>(J, 0, c);
  const double ny = *ey + tcs * (x0 - bx[pk] - z0 + bz[pi]) - dlt * aj_at<FIX>(J, 1, c);
  const double nz = *ez + tcs * (y0 - by[pi] - x0 + bx[pj]) - dlt * aj_at<FIX>(J, 2, c);
  *ex = nx;
  *ey = ny;
  *ez = nz;
}

// sum E^2 and B^2 over the cells 0..n-1: per-block partials, then one block
// adds them in a tree (deterministic)
constexpr int kFeBlocks = 256;

__global__ __launch_bounds__(kBlock) void k_field_energy_part(EbView v, double *part) {
  __shared__ double red[2][kBlock];
  const int64_t n = (int64_t)v.g.nx * v.g.ny * v.g.nz;
  double te = 0.0, tb = 0.0;
  for (int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x; o < n;
       o += (int64_t)kFeBlocks * kBlock) {
    int i, j, k;
    point_of(o, v.g.nx, v.g.ny, i, j, k);
    const double *q = v.eb + v.at(i, j, k);
    double p[6];
#pragma unroll
    for (int c = 0; c < 6; c++) p[c] = q[c * v.np];
    te = te + p[0] * p[0] + p[1] * p[1] + p[2] * p[2];
    tb = tb + p[BX] * p[BX] + p[BY] * p[BY] + p[BZ] * p[BZ];
  }
  red[0][threadIdx.x] = te;
  red[1][threadIdx.x] = tb;
  __syncthreads();
  for (int o = kBlock / 2; o > 0; o >>= 1) {
    if (threadIdx.x < (unsigned)o) {
      red[0][threadIdx.x] += red[0][threadIdx.x + o];
      red[1][threadIdx.x] += red[1][threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = red[0][0];
    part[2 * blockIdx.x + 1] = red[1][0];
  }
}

__global__ __launch_bounds__(kFeBlocks) void k_field_energy_final(const double *part, double cs,
                                                                  double vol, double *out,
                                                                  const int *dflag, int *hflag) {
  __shared__ double red[2][kFeBlocks];
  red[0][threadIdx.x] = part[2 * threadIdx.x];
  red[1][threadIdx.x] = part[2 * threadIdx.x + 1];
  __syncthreads();
  for (int o = kFeBlocks / 2; o > 0; o >>= 1) {
    if (threadIdx.x < (unsigned)o) {
      red[0][threadIdx.x] += red[0][threadIdx.x + o];
      red[1][threadIdx.x] += red[1][threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    out[0] = 0.5 * red[0][0] / vol;
    out[1] = 0.5 * cs * red[1][0] / vol;
    *hflag = *dflag;
  }
}

// copy the points [o0, o0 + n) of the box lo .. lo + ext - 1 of eb (inside the
// stored bounds) into records out(6, n)
__global__ __launch_bounds__(kBlock) void k_eb_box(EbView v, int lx, int ly, int lz, int ex, int ey,
                                                   int64_t o0, int64_t n, double *out) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= n) return;
  int i, j, k;
  point_of(o0 + o, ex, ey, i, j, k);
  const double *p = v.eb + v.at(i + lx, j + ly, k + lz);
  double2 *d = reinterpret_cast<double2 *>(out + o * 6);
#pragma unroll
  for (int q = 0; q < 3; q++) d[q] = make_double2(p[2 * q * v.np], p[(2 * q + 1) * v.np]);
}

unsigned blocks_of(const EbView &v) {
  return (unsigned)((v.np + kBlock - 1) / kBlock);
}

}  // namespace

EbView eb_view(const emg_ctx *c) {
  EbView v;
  v.eb = c->eb_dev;
  v.np = 1;
  for (int d = 0; d < 3; d++) {
    v.lo[d] = c->eb_lo[d];
    v.ext[d] = c->eb_ext[d];
    v.np *= c->eb_ext[d];
  }
  v.g = c->g;
  return v;
}

void launch_eb_split(emg_ctx *c, const double *rec, int64_t o0, int64_t n) {
  hipLaunchKernelGGL(k_eb_split, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, rec, eb_view(c), o0, n);
}

void launch_bfield(emg_ctx *c) {
  const EbView v = eb_view(c);
  hipLaunchKernelGGL(k_bfield, dim3(blocks_of(v)), dim3(kBlock), 0, c->stream, v);
}

void launch_efield(emg_ctx *c, double tcs, double dlt) {
  const EbView v = eb_view(c);
  CurrentView J;
  const bool fix = c->cfg.precision == EMG_FP32_FIXED;
  J.jacc = fix ? (const void *)c->jfx : (const void *)c->j64;
  for (int s = 0; s < EMG_MAX_SPECIES; s++) J.q[s] = c->cfg.q[s];
  J.nspec = c->sp.nspec;
  J.ncell = c->ncell;
  if (fix)
    hipLaunchKernelGGL(k_efield<true>, dim3(blocks_of(v)), dim3(kBlock), 0, c->stream, v, J, tcs,
                       dlt);
  else
    hipLaunchKernelGGL(k_efield<false>, dim3(blocks_of(v)), dim3(kBlock), 0, c->stream, v, J, tcs,
                       dlt);
}

void launch_eb_box(emg_ctx *c, const int lo[3], const int ext[3], int64_t o0, int64_t n,
                   double *out) {
  hipLaunchKernelGGL(k_eb_box, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, eb_view(c), lo[0], lo[1], lo[2], ext[0], ext[1], o0, n, out);
}

int64_t field_energy_part_need() { return 2 * kFeBlocks; }

void launch_field_energy(emg_ctx *c, double cs, double *part_dev, double *out) {
  const EbView v = eb_view(c);
  hipLaunchKernelGGL(k_field_energy_part, dim3(kFeBlocks), dim3(kBlock), 0, c->stream, v, part_dev);
  const double vol = (double)c->g.slx * c->g.sly * c->g.slz;
  hipLaunchKernelGGL(k_field_energy_final, dim3(1), dim3(kFeBlocks), 0, c->stream, part_dev, cs,
                     vol, out, c->dflag, c->hflag);
}

}  // namespace emg
