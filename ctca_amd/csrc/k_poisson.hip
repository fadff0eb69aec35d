// k_poisson.hip -- the electrostatic field solve on the device, for one
// periodic rank, so an ES step can stay on the device:
//   rho    = the deposited charge of every species + the background: the
//            per-node array of emg_set_background, if any, then the uniform
//            value (charge.F90:414-449 add_background_charge);
//   phi    : -lap7 phi = rho, spectrally: the 7-point Laplacian has the
//            eigenvalues kappa = sum_d (2 sin(pi k_d / n_d))^2
//            (inifft.F90:390-404), the zero mode is dropped
//            (poissn.F90:398-410); in three or five kernels of LDS lines where
//            they are faster, else real-to-complex FFTs from hipFFT;
//   E      = -grad phi on the staggered points (esfild.F90:351-367):
//            EX(i) = phi(i) - phi(i+1), etc., written into the device eb
//            (every point, ghosts as periodic images; B untouched) and, in
//            the same pass, relocated to the nodes (grdcrt); the nodes' B
//            stays unless eb's B has changed since it was relocated.
// The FFT round-off differs from FFTW's (which the reference uses); the solve
// is pinned by the spectral closed form and the 7-point residual.
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <new>
#include <string>

#include "emg_internal.h"
#include "fft_lines.h"

namespace emg {

constexpr int kPlaneThreads = 1024, kColumnThreads = 512;  // at most

struct EsSolver {
  hipfftHandle fwd = 0, inv = 0;
  bool have_fwd = false, have_inv = false;
  double *rho = nullptr;    // nz ny nx, then phi in place of it
  double2 *spec = nullptr;  // nz ny (nx/2 + 1)
  double *eig = nullptr;    // (2 sin(pi k / n))^2 of x, y, z: nx + ny + nz values
  int path = 0;             // SolvePath
  int kind = 0;             // of the axes' radices
  FftAxis *ax = nullptr;    // x, y, z
  double2 *tw = nullptr;    // e^(-2 pi i k / n) of x, y, z
};

namespace {

// Where the charge comes from: rho64 or rhofx of every species, and the
// background
struct RhoSum {
  const double *rho64;
  const unsigned long long *rhofx;
  int64_t ncell;
  const double *bkarr;
  double bk;
  int nspec;
  double q[EMG_MAX_SPECIES];
};

__device__ __forceinline__ double rho_total(const RhoSum &a, int64_t c) {
  auto of = [&](int s) {
    return a.rho64
               ? a.rho64[(int64_t)s * a.ncell + c]
               : a.q[s] *
                     ((double)(long long)a.rhofx[(int64_t)s * a.ncell + c] * (1.0 / kFixScale));
  };
  const double back = a.bkarr ? a.bkarr[c] : 0.0;
  double v = 0.0;
  int s = 0;
  for (; s + 1 < a.nspec; s += 2) {  // two loads in flight
    const double v0 = of(s), v1 = of(s + 1);
    v = v + v0 + v1;
  }
  if (s < a.nspec) v = v + of(s);
  if (a.bkarr) v = v + back;
  return v + a.bk;
}

__global__ __launch_bounds__(kBlock) void k_rho_total(RhoSum a, double *out) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c < a.ncell) out[c] = rho_total(a, c);
}

// the eigenvalues of every axis, once per context (three sines per mode and solve
// made the division take 24 us on 256 x 256 x 64 cells, 13 now).  By the smaller
// of k and n - k: near half a turn a sine loses its low bits, which the largest
// modes of phi then lack.
__global__ __launch_bounds__(kBlock) void k_poisson_eig(double *eig, Grid g) {
  const int o = blockIdx.x * kBlock + threadIdx.x;
  if (o >= g.nx + g.ny + g.nz) return;
  const int k = o < g.nx ? o : (o < g.nx + g.ny ? o - g.nx : o - g.nx - g.ny);
  const int n = o < g.nx ? g.nx : (o < g.nx + g.ny ? g.ny : g.nz);
  const double s = 2.0 * sinpi((double)min(k, n - k) / n);
  eig[o] = s * s;
}

// spectrum / (N kappa), the zero mode set to 0 (N: the inverse transform is
// unnormalised)
__global__ __launch_bounds__(kBlock) void k_poisson_divide(double2 *spec,
                                                           const double *__restrict__ eig, Grid g) {
  const int hx = g.nx / 2 + 1;
  const int64_t n = (int64_t)g.nz * g.ny * hx;
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= n) return;
  int kx, ky, kz;
  point_of(o, hx, g.ny, kx, ky, kz);
  const double kappa = eig[g.nx + g.ny + kz] + eig[g.nx + ky] + eig[kx];
  double2 v = spec[o];
  if (o == 0) {
    v.x = 0.0;
    v.y = 0.0;
  } else {
    const double f = 1.0 / (kappa * ((double)g.nx * g.ny * g.nz));
    v.x *= f;
    v.y *= f;
  }
  spec[o] = v;
}

// e^(-2 pi i k / n) of every axis, the angle folded to at most an eighth of a
// turn by whole numbers first, so that only the sine and cosine round
__global__ __launch_bounds__(kBlock) void k_poisson_twiddle(double2 *tw, Grid g, FftAxis x,
                                                            FftAxis y, FftAxis z, FftAxis *ax) {
  const int o = blockIdx.x * kBlock + threadIdx.x;
  if (o == 0) {
    ax[0] = x;
    ax[1] = y;
    ax[2] = z;
  }
  if (o >= g.nx + g.ny + g.nz) return;
  const int k = o < g.nx ? o : (o < g.nx + g.ny ? o - g.nx : o - g.nx - g.ny);
  const int n = o < g.nx ? g.nx : (o < g.nx + g.ny ? g.ny : g.nz);
  const int quarter = (8 * k + n) / (2 * n);  // the nearest quarter turn
  double s, c;
  sincospi(0.5 * (4 * k - quarter * n) / n, &s, &c);
  switch (quarter & 3) {
    case 0: tw[o] = make_double2(c, -s); break;
    case 1: tw[o] = make_double2(-s, -c); break;
    case 2: tw[o] = make_double2(-c, s); break;
    default: tw[o] = make_double2(s, c);
  }
}

// The solve of a small grid in three kernels, the lines of which stay in LDS:
// the charge of an x-y plane and its transform, every (kx, ky) column's
// transform, division and inverse, and the planes' inverse.  hipFFT's four
// kernels, the charge sum and the division moved each value six times through
// launches of 3 to 6 us that do little work.  A block's time is its chain of
// latencies (16^3 cells: three kernels of 5 us): its tables and its data are
// loaded together, it has a thread per element where that is at most 1024, and
// each kernel holds the code of its radices only.
struct PlaneArgs {
  const FftAxis *ax;
  const double2 *tw;
  int ny, rows;        // rows per block: a whole plane, or some of its x lines
  FastDiv nx, np, hx;  // np: pairs of x lines
  int stride, buf;     // of the pairs (odd: no bank conflicts); elements per buffer
};
constexpr int kAxisWords = sizeof(FftAxis) / 4;

// one axis' passes; the result's buffer comes back in x
template <bool INV, int KIND>
__device__ __forceinline__ void fft_axis_lines(const FftAxis &a, double2 *&x, double2 *&y,
                                               const FastDiv &lines, int stride,
                                               const double2 *tw) {
  const int npass = __builtin_amdgcn_readfirstlane(a.npass);
  for (int p = 0; p < npass; p++) {
    fft_pass_of<INV, KIND>(a, p, x, y, lines, stride, tw, threadIdx.x, blockDim.x);
    __syncthreads();
    double2 *z = x;
    x = y;
    y = z;
  }
}

extern __shared__ double2 fft_lds[];

// put(t, get(t)) for this thread's t < n, U loads in flight
template <int U, class Get, class Put>
__device__ __forceinline__ void stage(int n, Get get, Put put) {
  const int nt = blockDim.x;
  for (int t0 = threadIdx.x; t0 < n; t0 += U * nt) {
    double2 v[U];
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t0 + u * nt < n) v[u] = get(t0 + u * nt);
#pragma unroll
    for (int u = 0; u < U; u++)
      if (t0 + u * nt < n) put(t0 + u * nt, v[u]);
  }
}

// The tables of a block, n axes' and m twiddles, on their way to LDS: get()
// issues the loads, put() (after the loads of the data) stores, so that one
// memory latency covers all.  Blocks have at least 2 kAxisWords threads.
struct Tables {
  int word;
  double2 w;
  __device__ __forceinline__ void get(const FftAxis *ax, int n, const double2 *tw, int m) {
    const int tid = threadIdx.x;
    if (tid < n * kAxisWords) word = reinterpret_cast<const int *>(ax)[tid];
    if (tid < m) w = tw[tid];
  }
  __device__ __forceinline__ void put(FftAxis *ax, int n, const double2 *tw, double2 *out, int m) {
    const int tid = threadIdx.x;
    if (tid < n * kAxisWords) reinterpret_cast<int *>(ax)[tid] = word;
    if (tid < m) out[tid] = w;
    for (int q = tid + blockDim.x; q < m; q += blockDim.x) out[q] = tw[q];
  }
};

// YAXIS: the block's rows are a whole plane, which goes through y as well
template <int KIND, bool YAXIS>
__global__ __launch_bounds__(kPlaneThreads) void k_plane_forward(PlaneArgs a, RhoSum rho,
                                                                 double2 *spec) {
  __shared__ FftAxis ax[2];
  double2 *x = fft_lds, *y = x + a.buf, *tw = y + a.buf;
  const int nx = a.nx.d, tid = threadIdx.x, nt = blockDim.x;
  const int naxes = YAXIS ? 2 : 1, ntw = YAXIS ? nx + a.ny : nx;
  const int row0 = YAXIS ? 0 : blockIdx.y * a.rows, ny = YAXIS ? a.ny : min(a.rows, a.ny - row0);
  const int64_t line0 = (int64_t)blockIdx.x * a.ny + row0;
  Tables tab;
  tab.get(a.ax, naxes, a.tw, ntw);
  stage<1>(
      nx * a.np.d,
      [&](int t) {
        const int p = div(t, a.nx), i = t - p * nx;
        const int64_t c = (line0 + min(2 * p, ny - 1)) * nx + i;
        const double v = rho_total(rho, 2 * p + 1 < ny ? c + nx : c);
        return make_double2(rho_total(rho, c), 2 * p + 1 < ny ? v : 0.0);
      },
      [&](int t, double2 v) {
        const int p = div(t, a.nx), i = t - p * nx;
        x[i * a.stride + p] = v;
      });
  tab.put(ax, naxes, a.tw, tw, ntw);
  __syncthreads();
  fft_axis_lines<false, KIND>(ax[0], x, y, a.np, a.stride, tw);
  split_pairs(x, a.stride, y, nx, ny, a.np, tid, nt);
  __syncthreads();
  if (YAXIS) fft_axis_lines<false, KIND>(ax[1], y, x, a.hx, a.hx.d, tw + nx);
  const int n = a.hx.d * ny;
  double2 *out = spec + line0 * a.hx.d;
  for (int t = tid; t < n; t += nt) out[t] = y[t];
}

template <int KIND, bool YAXIS>
__global__ __launch_bounds__(kPlaneThreads) void k_plane_inverse(PlaneArgs a, const double2 *spec,
                                                                 double *phi) {
  __shared__ FftAxis ax[2];
  double2 *x = fft_lds, *y = x + a.buf, *tw = y + a.buf;
  const int nx = a.nx.d, tid = threadIdx.x, nt = blockDim.x;
  const int naxes = YAXIS ? 2 : 1, ntw = YAXIS ? nx + a.ny : nx;
  const int row0 = YAXIS ? 0 : blockIdx.y * a.rows, ny = YAXIS ? a.ny : min(a.rows, a.ny - row0);
  const int64_t line0 = (int64_t)blockIdx.x * a.ny + row0;
  Tables tab;
  tab.get(a.ax, naxes, a.tw, ntw);
  const double2 *in = spec + line0 * a.hx.d;
  stage<4>(a.hx.d * ny, [&](int t) { return in[t]; }, [&](int t, double2 v) { x[t] = v; });
  tab.put(ax, naxes, a.tw, tw, ntw);
  __syncthreads();
  if (YAXIS) fft_axis_lines<true, KIND>(ax[1], x, y, a.hx, a.hx.d, tw + nx);
  join_pairs(x, y, a.stride, nx, ny, a.np, tid, nt);
  __syncthreads();
  fft_axis_lines<true, KIND>(ax[0], y, x, a.np, a.stride, tw);
  for (int t = tid; t < nx * a.np.d; t += nt) {
    const int p = div(t, a.nx), i = t - p * nx;
    const double2 v = y[i * a.stride + p];
    const int64_t c = (line0 + 2 * p) * nx + i;
    if (2 * p < ny) phi[c] = v.x;
    if (2 * p + 1 < ny) phi[c + nx] = v.y;
  }
}

// The transforms of kColumns neighbouring columns per block (128 bytes of each
// of their elements): of z, with the division and the inverse (SOLVE), or of y
// one way.  Element k of column c of part blockIdx.y is spec[part y + k ncol + c].
constexpr int kColumns = 8;
enum ColumnMode { kForward, kInverse, kSolve };
struct ColumnArgs {
  const FftAxis *ax;
  const double2 *tw;
  int n, ncol;
  int64_t part;
  const double *ez, *ey, *ex;  // kSolve: the eigenvalues
  int hx;
  double cells;
};
template <int KIND, ColumnMode MODE>
__global__ __launch_bounds__(kColumnThreads) void k_columns(ColumnArgs a, double2 *spec) {
  __shared__ FftAxis ax;
  const int col0 = blockIdx.x * kColumns, n = a.n, nt = blockDim.x, tid = threadIdx.x;
  double2 *x = fft_lds, *y = x + n * kColumns, *tw = y + n * kColumns;
  double *ez = reinterpret_cast<double *>(tw + n);
  // a thread's column is the same all through (nt is a multiple of kColumns)
  const int l = tid % kColumns, col = min(col0 + l, a.ncol - 1);
  const bool mine = col0 + l < a.ncol;
  Tables tab;
  tab.get(a.ax, 1, a.tw, n);
  double e0 = 0.0, ey = 0.0, ex = 0.0;
  if (MODE == kSolve) {
    const int ky = col / a.hx, kx = col - ky * a.hx;
    if (tid < n) e0 = a.ez[tid];
    ey = a.ey[ky];
    ex = a.ex[kx];
  }
  double2 *own = spec + blockIdx.y * a.part + col;
  stage<4>(
      n * kColumns, [&](int t) { return own[(int64_t)(t / kColumns) * a.ncol]; },
      [&](int t, double2 v) { x[t] = v; });
  tab.put(&ax, 1, a.tw, tw, n);
  if (MODE == kSolve) {
    if (tid < n) ez[tid] = e0;
    for (int q = tid + nt; q < n; q += nt) ez[q] = a.ez[q];
  }
  __syncthreads();
  const FastDiv cols{(uint32_t)((1ull << 32) / kColumns), kColumns};
  fft_axis_lines<MODE == kInverse, KIND>(ax, x, y, cols, kColumns, tw);
  if (MODE == kSolve) {
    for (int t = tid; t < n * kColumns; t += nt) {
      const double kappa = ez[t / kColumns] + ey + ex;
      double2 v = x[t];
      if (col == 0 && t < kColumns) {
        v.x = 0.0;
        v.y = 0.0;
      } else {
        const double f = 1.0 / (kappa * a.cells);
        v.x *= f;
        v.y *= f;
      }
      x[t] = v;
    }
    __syncthreads();
    fft_axis_lines<true, KIND>(ax, x, y, cols, kColumns, tw);
  }
  if (mine)
    for (int t = tid; t < n * kColumns; t += nt) own[(int64_t)(t / kColumns) * a.ncol] = x[t];
}

// E = -grad phi at every point of eb, and at the nodes 0..n its relocation
// (k_relocate's expression on the same differences) with the uniform e0.  One
// pass over phi instead of a pass that writes eb and one that reads all of eb
// back: 228 -> 52 us on 256 x 256 x 64 cells (FP32 nodes).
__global__ __launch_bounds__(kBlock) void k_es_efield(const double *__restrict__ phi, EbView v,
                                                      double *__restrict__ node64,
                                                      float *__restrict__ node32, int64_t ncell,
                                                      double e0x, double e0y, double e0z) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o >= v.np) return;
  const Grid &g = v.g;
  int i, j, k;
  point_of(o, v.ext[0], v.ext[1], i, j, k);
  i += v.lo[0];
  j += v.lo[1];
  k += v.lo[2];
  const int ci = periodic_index(i, g.nx), cj = periodic_index(j, g.ny),
            ck = periodic_index(k, g.nz);
  const int64_t sy = g.nx, sz = (int64_t)g.nx * g.ny, c = ck * sz + cj * sy + ci;
  const double p0 = phi[c];
  const double ex = p0 - phi[ci + 1 == g.nx ? c - ci : c + 1],
               ey = p0 - phi[cj + 1 == g.ny ? c - cj * sy : c + sy],
               ez = p0 - phi[ck + 1 == g.nz ? c - ck * sz : c + sz];
  v.eb[o] = ex;
  v.eb[v.np + o] = ey;
  v.eb[2 * v.np + o] = ez;
  const int last = node32 ? 1 : 0;  // FP32 nodes end at n - 1
  if (i < 0 || j < 0 || k < 0 || i > g.nx - last || j > g.ny - last || k > g.nz - last) return;
  const double nx = 0.5 * (ex + (phi[ci == 0 ? c + g.nx - 1 : c - 1] - p0)) + e0x,
               ny = 0.5 * (ey + (phi[cj == 0 ? c + sz - sy : c - sy] - p0)) + e0y,
               nz = 0.5 * (ez + (phi[ck == 0 ? c + (g.nz - 1) * sz : c - sz] - p0)) + e0z;
  if (node64) {
    double *d = node64 + 8 * (((int64_t)k * (g.ny + 1) + j) * (g.nx + 1) + i);
    *reinterpret_cast<double2 *>(d) = make_double2(nx, ny);
    d[2] = nz;
  } else {
    reinterpret_cast<float4 *>(node32)[c] = make_float4((float)nx, (float)ny, (float)nz, 0.f);
  }
}

}  // namespace

constexpr size_t kPlaneLds = 159 * 1024;  // of 160 KB, less the static part
constexpr int kLargestRadix = 211;        // (a prime r costs r / 2 products per element)
constexpr int kLongestLine = 512;         // (two buffers of 8 columns in LDS)
// kLines: pairs of x lines per block, of about kRowElems elements.  (199x40x40
// cells 78 us with 256 threads, 61 with 512; 2048 elements 82.)
constexpr int kRowElems = 1024, kRowThreads = 512;
// a thread per element where they fit
static int threads_for(int elems, int most) {
  return std::min(most, std::max(128, (elems + 63) / 64 * 64));
}

static int fft_check(hipfftResult r, const char *what) {
  if (r == HIPFFT_SUCCESS) return EMG_OK;
  return set_error(EMG_ERR_HIP, std::string(what) + ": hipFFT error " + std::to_string((int)r));
}

void es_solver_free(emg_ctx *c) {
  EsSolver *s = c->es;
  if (!s) return;
  if (s->have_fwd) (void)hipfftDestroy(s->fwd);
  if (s->have_inv) (void)hipfftDestroy(s->inv);
  if (s->rho) (void)hipFree(s->rho);
  if (s->spec) (void)hipFree(s->spec);
  if (s->eig) (void)hipFree(s->eig);
  if (s->tw) (void)hipFree(s->tw);
  if (s->ax) (void)hipFree(s->ax);
  delete s;
  c->es = nullptr;
}

// How the field solve runs: kPlanes as above; kLines with x and y in kernels of
// their own (five kernels, for planes that LDS does not hold); kLibrary
enum SolvePath { kLibrary, kPlanes, kLines };

// rows per block, elements per buffer, and LDS bytes of k_plane_*
static int plane_rows(const Grid &g, SolvePath path) {
  return path == kPlanes ? g.ny : std::min((g.ny + 1) / 2 * 2, 2 * std::max(1, kRowElems / g.nx));
}
static int plane_elems(const Grid &g, SolvePath path) {
  const int rows = plane_rows(g, path), np = (rows + 1) / 2;
  return std::max(g.nx * (np | 1), rows * (g.nx / 2 + 1));
}
static size_t plane_lds(const Grid &g, SolvePath path) {
  return sizeof(double2) *
         (2 * (size_t)plane_elems(g, path) + g.nx + (path == kPlanes ? g.ny : 0));
}
static size_t column_lds(int n) {
  return (sizeof(double2) * (2 * kColumns + 1) + sizeof(double)) * (size_t)n;
}

// Which one is the fastest.  Solve, E included, hipFFT : planes : lines in us.
// Small planes: 16^3 cells 19.3 : 17.7 : 22.0, 32^3 22.3 : 19.4 : 24.1, 64^3 36.7 :
// 29.9 : 36.4, 64x64x4 26.7 : 22.2 : 24.8.  Above 3000 elements a plane is a long
// chain for its one block, which pays where there are many: 90x100 cells by 4 27.6
// : 36.4 : 28.5, by 32 41.7 : 44.8 : 39.6, by 48 52.5 : 48.9 : 46.7, by 96 75.5 :
// 56.9 : 63.9; 84x84 by 4 34 : 32 : 29, by 48 48 : 44 : 46; 60x140 by 4 52 : 35 : 30,
// by 48 65 : 51 : 52; 90x70x51 46.8 : 44.9 : 46.5; 96^3 73 : 54 : 63.
// From a prime factor of 19 on hipFFT changes to a longer algorithm, and the lines
// do the work of the larger planes: 31^3 117 : 23 : 28, 53^3 150 : 36 : 43, 62^3
// 128 : 38 : 38, 101x40x40 74 : 38 : 40, 95x66x40 87 : 43 : 38, 97x98x50 113 : 78 : 62,
// 114x95x133 252 : - : 112, 191x181x173 1141 : - : 596.
// An odd nx costs hipFFT's real transforms about twice an even one, and the lines
// nothing: 105x100x100 131 : - : 88, 125^3 154 : - : 99, 225^3 1204 : - : 503.
// Else, with factors 2, 3 and 5, the lines up to some 2 million cells (100x100x16
// 49 : - : 33, 100^3 83 : - : 69, 48x200x96 80 : - : 63, 128^3 117 : - : 106, 256x64x96
// 110 : - : 90, but 512x64x64 111 : - : 118), beyond that about equal (150^3 155 : - :
// 152, 160^3 169 : - : 170, 256x256x64 194 : - : 200); with 7, 11 or 13 now this, now
// that (110^3 106 : - : 99, 126^3 127 : - : 109, 112^3 94 : - : 102, 98x112x112 84 : -
// : 94, 154x143x91 124 : - : 135, 180x150x170 219 : - : 251).
// The first solve of planes and lines also has no kernels to compile at run time
// (1.6 s : 0.2 ms).
static SolvePath solve_path(const Grid &g, FftAxis ax[3]) {
  const int n[3] = {g.nx, g.ny, g.nz};
  int largest = 0, kind = 0;
  for (int d = 0; d < 3; d++) {
    if (n[d] > kLongestLine || !fft_axis(n[d], kLargestRadix, &ax[d])) return kLibrary;
    kind = std::max(kind, radix_kind(ax[d]));
    for (int p = 0; p < ax[d].npass; p++) largest = std::max(largest, ax[d].r[p]);
  }
  if (plane_lds(g, kPlanes) <= kPlaneLds)
    return plane_elems(g, kPlanes) <= 3000 || (largest < 19 && g.nz >= 48) ? kPlanes : kLines;
  if (largest >= 19 || g.nx % 2) return kLines;
  const bool small = (int64_t)g.nx * g.ny * g.nz <= 1 << 21 && std::max({n[0], n[1], n[2]}) < 512;
  return kind < 2 && small ? kLines : kLibrary;
}

template <class F>
static void with_kind(int kind, F f) {
  if (kind == 0)
    f(std::integral_constant<int, 0>());
  else if (kind == 1)
    f(std::integral_constant<int, 1>());
  else
    f(std::integral_constant<int, 2>());
}

// the plans keep the stream they are given: again when the context's changes
int es_solver_stream(emg_ctx *c) {
  EsSolver *s = c->es;
  int rc = EMG_OK;
  if (s && s->have_fwd) rc = fft_check(hipfftSetStream(s->fwd, c->stream), "set stream");
  if (!rc && s && s->have_inv) rc = fft_check(hipfftSetStream(s->inv, c->stream), "set stream");
  return rc;
}

static int es_fft_plans(emg_ctx *c, EsSolver *s) {
  int rc = fft_check(hipfftPlan3d(&s->fwd, c->g.nz, c->g.ny, c->g.nx, HIPFFT_D2Z), "plan D2Z");
  if (!rc) s->have_fwd = true;
  if (!rc) rc = fft_check(hipfftPlan3d(&s->inv, c->g.nz, c->g.ny, c->g.nx, HIPFFT_Z2D), "plan Z2D");
  if (!rc) s->have_inv = true;
  return rc ? rc : es_solver_stream(c);
}

static int es_solver_get(emg_ctx *c, EsSolver **out) {
  if (c->es) {
    *out = c->es;
    return EMG_OK;
  }
  EsSolver *s = new (std::nothrow) EsSolver();
  if (!s) return set_error(EMG_ERR_NOMEM, "field solver");
  c->es = s;
  const int64_t hx = c->g.nx / 2 + 1;
  const int neig = c->g.nx + c->g.ny + c->g.nz;
  int rc = EMG_OK;
  if (!dev_malloc(c, &s->rho, sizeof(double) * c->ncell) ||
      !dev_malloc(c, &s->spec, sizeof(double2) * c->g.nz * c->g.ny * hx) ||
      !dev_malloc(c, &s->eig, sizeof(double) * neig))
    rc = set_error(EMG_ERR_NOMEM, "field solver arrays");
  FftAxis ax[3];
  s->path = solve_path(c->g, ax);
  if (!rc && s->path != kLibrary) {
    if (!dev_malloc(c, &s->tw, sizeof(double2) * neig) ||
        !dev_malloc(c, &s->ax, sizeof(ax)))
      rc = set_error(EMG_ERR_NOMEM, "field solver arrays");
    for (int d = 0; d < 3; d++) s->kind = std::max(s->kind, radix_kind(ax[d]));
    auto allow = [&](auto kernel) {
      if (!rc)
        rc = hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)kPlaneLds),
                       "field solver LDS");
    };
    with_kind(s->kind, [&](auto kind) {
      constexpr int K = decltype(kind)::value;
      if (s->path == kPlanes) {
        allow(k_plane_forward<K, true>);
        allow(k_plane_inverse<K, true>);
      } else {
        allow(k_plane_forward<K, false>);
        allow(k_plane_inverse<K, false>);
        allow(k_columns<K, kForward>);
        allow(k_columns<K, kInverse>);
      }
      allow(k_columns<K, kSolve>);
    });
  }
  if (!rc && s->path == kLibrary) rc = es_fft_plans(c, s);
  if (rc) {
    es_solver_free(c);
    return rc;
  }
  const dim3 ge((unsigned)((neig + kBlock - 1) / kBlock));
  hipLaunchKernelGGL(k_poisson_eig, ge, dim3(kBlock), 0, c->stream, s->eig, c->g);
  if (s->path != kLibrary)
    hipLaunchKernelGGL(k_poisson_twiddle, ge, dim3(kBlock), 0, c->stream, s->tw, c->g, ax[0], ax[1],
                       ax[2], s->ax);
  *out = s;
  return EMG_OK;
}
static void plane_solve(emg_ctx *c, EsSolver *s, const RhoSum &sum) {
  const Grid &g = c->g;
  const SolvePath path = (SolvePath)s->path;
  const int hx = g.nx / 2 + 1, rows = plane_rows(g, path), np = (rows + 1) / 2;
  const PlaneArgs a{s->ax, s->tw, g.ny, rows, fast_div(g.nx), fast_div(np), fast_div(hx), np | 1,
                    plane_elems(g, path)};
  const ColumnArgs az{s->ax + 2,
                      s->tw + g.nx + g.ny,
                      g.nz,
                      hx * g.ny,
                      0,
                      s->eig + g.nx + g.ny,
                      s->eig + g.nx,
                      s->eig,
                      hx,
                      (double)g.nx * g.ny * g.nz};
  const ColumnArgs ay{s->ax + 1, s->tw + g.nx, g.ny,    hx,  (int64_t)hx * g.ny,
                      nullptr,   nullptr,      nullptr, hx, 0.0};
  const size_t lp = plane_lds(g, path);
  const dim3 gp(g.nz, (g.ny + rows - 1) / rows), gz((az.ncol + kColumns - 1) / kColumns),
      gy((hx + kColumns - 1) / kColumns, g.nz);
  const dim3 tp(threads_for(g.nx * np, path == kPlanes ? kPlaneThreads : kRowThreads)),
      ty(threads_for(g.ny * kColumns, kColumnThreads)),
      tz(threads_for(g.nz * kColumns, kColumnThreads));
  with_kind(s->kind, [&](auto kind) {
    constexpr int K = decltype(kind)::value;
    auto columns = [&](auto kernel, dim3 grid, dim3 threads, const ColumnArgs &ca) {
      hipLaunchKernelGGL(kernel, grid, threads, column_lds(ca.n), c->stream, ca, s->spec);
    };
    if (path == kPlanes) {
      hipLaunchKernelGGL((k_plane_forward<K, true>), gp, tp, lp, c->stream, a, sum, s->spec);
      columns(k_columns<K, kSolve>, gz, tz, az);
      hipLaunchKernelGGL((k_plane_inverse<K, true>), gp, tp, lp, c->stream, a, s->spec, s->rho);
    } else {
      hipLaunchKernelGGL((k_plane_forward<K, false>), gp, tp, lp, c->stream, a, sum, s->spec);
      columns(k_columns<K, kForward>, gy, ty, ay);
      columns(k_columns<K, kSolve>, gz, tz, az);
      columns(k_columns<K, kInverse>, gy, ty, ay);
      hipLaunchKernelGGL((k_plane_inverse<K, false>), gp, tp, lp, c->stream, a, s->spec, s->rho);
    }
  });
}

static int fft_solve(emg_ctx *c, EsSolver *s, const RhoSum &sum) {
  const unsigned gc = (unsigned)((c->ncell + kBlock - 1) / kBlock);
  hipLaunchKernelGGL(k_rho_total, dim3(gc), dim3(kBlock), 0, c->stream, sum, s->rho);
  int rc = fft_check(hipfftExecD2Z(s->fwd, s->rho, reinterpret_cast<hipfftDoubleComplex *>(s->spec)),
                     "D2Z");
  if (rc) return rc;
  const int64_t ns = (int64_t)c->g.nz * c->g.ny * (c->g.nx / 2 + 1);
  hipLaunchKernelGGL(k_poisson_divide, dim3((unsigned)((ns + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, c->stream, s->spec, s->eig, c->g);
  return fft_check(hipfftExecZ2D(s->inv, reinterpret_cast<hipfftDoubleComplex *>(s->spec), s->rho),
                   "Z2D");
}

int solve_es(emg_ctx *c, double rhobk) {
  EsSolver *s = nullptr;
  int rc = es_solver_get(c, &s);
  if (rc) return rc;
  const bool fix = c->cfg.precision == EMG_FP32_FIXED;
  RhoSum sum{fix ? nullptr : c->rho64, fix ? c->rhofx : nullptr, c->ncell, c->bk_dev, rhobk,
             c->sp.nspec, {}};
  for (int k = 0; k < c->sp.nspec; k++) sum.q[k] = c->sp.q[k];
  if (s->path != kLibrary)
    plane_solve(c, s, sum);
  else
    rc = fft_solve(c, s, sum);
  if (rc) return rc;
  const EbView v = eb_view(c);
  timer_begin(c, kTRelocate);
  hipLaunchKernelGGL(k_es_efield, dim3((unsigned)((v.np + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, s->rho, v, fix ? nullptr : c->node64, fix ? c->node32 : nullptr,
                     c->ncell, c->cfg.e0[0], c->cfg.e0[1], c->cfg.e0[2]);
  timer_end(c, kTRelocate);
  // the nodes' B as well where it may be another one; always in a recorded solve,
  // which may be replayed after a B update that this call cannot know of
  if (!c->nodes_b_valid || c->b_recorded || capturing(c)) launch_relocate64(c);
  return hip_check(hipGetLastError(), "field solve launch");
}

int read_potential(emg_ctx *c, double *phi) {
  if (!c->es) return set_error(EMG_ERR_STATE, "no field solve yet");
  // (the particles' errors are left to the calls on them)
  return io_read_array(c, phi, c->es->rho, sizeof(double) * c->ncell, false);
}

}  // namespace emg
