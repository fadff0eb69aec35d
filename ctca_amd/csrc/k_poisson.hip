// k_poisson.hip -- the electrostatic field solve on the device, for one
// periodic rank, so an ES step can stay on the device:
//   rho    = the deposited charge of every species + the background: the
//            per-node array of emg_set_background, if any, then the uniform
//            value (charge.F90:414-449 add_background_charge);
//   phi    : -lap7 phi = rho, spectrally: the 7-point Laplacian has the
//            eigenvalues kappa = sum_d (2 sin(pi k_d / n_d))^2
//            (inifft.F90:390-404), the zero mode is dropped
//            (poissn.F90:398-410); real-to-complex FFTs from hipFFT;
//   E      = -grad phi on the staggered points (esfild.F90:351-367):
//            EX(i) = phi(i) - phi(i+1), etc., written into the device eb
//            (every point, ghosts as periodic images; B untouched) and, in
//            the same pass, relocated to the nodes (grdcrt); the nodes' B
//            stays unless eb's B has changed since it was relocated.
// The FFT round-off differs from FFTW's (which the reference uses); the solve
// is pinned by the spectral closed form and the 7-point residual.
#include <hipfft/hipfft.h>

#include <cmath>
#include <new>
#include <string>

#include "emg_internal.h"

namespace emg {

struct EsSolver {
  hipfftHandle fwd = 0, inv = 0;
  bool have_fwd = false, have_inv = false;
  double *rho = nullptr;    // nz ny nx, then phi in place of it
  double2 *spec = nullptr;  // nz ny (nx/2 + 1)
  double *eig = nullptr;    // (2 sin(pi k / n))^2 of x, y, z: nx + ny + nz values
};

namespace {

__global__ __launch_bounds__(kBlock) void k_rho_total(const double *rho64,
                                                      const unsigned long long *rhofx,
                                                      SpeciesTab sp, int64_t ncell,
                                                      const double *bkarr, double bk,
                                                      double *out) {
  const int64_t c = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (c >= ncell) return;
  double v = 0.0;
  for (int s = 0; s < sp.nspec; s++) {
    if (rho64)
      v = v + rho64[(int64_t)s * ncell + c];
    else
      v = v + sp.q[s] * ((double)(long long)rhofx[(int64_t)s * ncell + c] * (1.0 / kFixScale));
  }
  if (bkarr) v = v + bkarr[c];
  out[c] = v + bk;
}

// the eigenvalues of every axis, once per context (three sines per mode and solve
// made the division take 24 us on 256 x 256 x 64 cells, 13 now)
__global__ __launch_bounds__(kBlock) void k_poisson_eig(double *eig, Grid g) {
  const int o = blockIdx.x * kBlock + threadIdx.x;
  if (o >= g.nx + g.ny + g.nz) return;
  const int k = o < g.nx ? o : (o < g.nx + g.ny ? o - g.nx : o - g.nx - g.ny);
  const int n = o < g.nx ? g.nx : (o < g.nx + g.ny ? g.ny : g.nz);
  const double s = 2.0 * sin(3.141592653589793 * k / n);
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
  delete s;
  c->es = nullptr;
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
  if (hipMalloc(&s->rho, sizeof(double) * c->ncell) != hipSuccess ||
      hipMalloc(&s->spec, sizeof(double2) * c->g.nz * c->g.ny * hx) != hipSuccess ||
      hipMalloc(&s->eig, sizeof(double) * neig) != hipSuccess)
    rc = set_error(EMG_ERR_NOMEM, "field solver arrays");
  if (!rc) rc = fft_check(hipfftPlan3d(&s->fwd, c->g.nz, c->g.ny, c->g.nx, HIPFFT_D2Z), "plan D2Z");
  if (!rc) s->have_fwd = true;
  if (!rc) rc = fft_check(hipfftPlan3d(&s->inv, c->g.nz, c->g.ny, c->g.nx, HIPFFT_Z2D), "plan Z2D");
  if (!rc) s->have_inv = true;
  if (!rc) rc = fft_check(hipfftSetStream(s->fwd, c->stream), "set stream");
  if (!rc) rc = fft_check(hipfftSetStream(s->inv, c->stream), "set stream");
  if (rc) {
    es_solver_free(c);
    return rc;
  }
  hipLaunchKernelGGL(k_poisson_eig, dim3((unsigned)((neig + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, s->eig, c->g);
  *out = s;
  return EMG_OK;
}

int solve_es(emg_ctx *c, double rhobk) {
  EsSolver *s = nullptr;
  int rc = es_solver_get(c, &s);
  if (rc) return rc;
  const unsigned gc = (unsigned)((c->ncell + kBlock - 1) / kBlock);
  const bool fix = c->cfg.precision == EMG_FP32_FIXED;
  hipLaunchKernelGGL(k_rho_total, dim3(gc), dim3(kBlock), 0, c->stream, fix ? nullptr : c->rho64,
                     fix ? c->rhofx : nullptr, c->sp, c->ncell, c->bk_dev, rhobk, s->rho);
  rc = fft_check(hipfftExecD2Z(s->fwd, s->rho, reinterpret_cast<hipfftDoubleComplex *>(s->spec)),
                 "D2Z");
  if (rc) return rc;
  const int64_t ns = (int64_t)c->g.nz * c->g.ny * (c->g.nx / 2 + 1);
  hipLaunchKernelGGL(k_poisson_divide, dim3((unsigned)((ns + kBlock - 1) / kBlock)), dim3(kBlock),
                     0, c->stream, s->spec, s->eig, c->g);
  rc = fft_check(hipfftExecZ2D(s->inv, reinterpret_cast<hipfftDoubleComplex *>(s->spec), s->rho),
                 "Z2D");
  if (rc) return rc;
  const EbView v = eb_view(c);
  timer_begin(c, kTRelocate);
  hipLaunchKernelGGL(k_es_efield, dim3((unsigned)((v.np + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                     c->stream, s->rho, v, fix ? nullptr : c->node64, fix ? c->node32 : nullptr,
                     c->ncell, c->cfg.e0[0], c->cfg.e0[1], c->cfg.e0[2]);
  timer_end(c, kTRelocate);
  if (!c->nodes_b_valid) launch_relocate64(c);
  return hip_check(hipGetLastError(), "field solve launch");
}

int read_potential(emg_ctx *c, double *phi) {
  if (!c->es) return set_error(EMG_ERR_STATE, "no field solve yet");
  return io_read_array(c, phi, c->es->rho, sizeof(double) * c->ncell);
}

}  // namespace emg
