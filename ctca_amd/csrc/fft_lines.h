// fft_lines.h -- complex FP64 Fourier transforms of many short lines that lie
// in one block's LDS, and the real <-> complex steps around them, for the field
// solve of small grids (k_poisson.hip).
//
// Element i of line l is buf[i * stride + l]: neighbouring threads take
// neighbouring lines, so their accesses fall on different banks whatever the
// radix.  A pass reads one buffer and writes the other (the self-sorting form that
// Cochran et al. 1967 credit to Stockham: no bit reversal).  With ns the product of
// the radices done, pass r takes for j = 0 .. n/r - 1, k = j mod ns, the inputs x[j
// + p n/r] times w^(p k n / (ns r)), w = e^(-2 pi i / n), transforms those r
// values, and writes result q to (j / ns) ns r + k + q ns.
//
// Radices 2, 3, 4, 5, 7, 8, 11 and 13 transform in registers; any other prime sums
// its products straight from LDS, and comes first (ns = 1, no twiddles), where
// results q and r - q share theirs.
//
// The functions do the work of thread tid of nt; the caller separates them with
// barriers.
#ifndef EMG_FFT_LINES_H
#define EMG_FFT_LINES_H

#include <hip/hip_runtime.h>

#include <type_traits>

namespace emg {

constexpr int kMaxPasses = 8;

// q = t / d for t d < 2^32
struct FastDiv {
  uint32_t m;
  int d;
};
inline FastDiv fast_div(int d) {
  return FastDiv{d == 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d), d};
}
__host__ __device__ inline int div(int t, const FastDiv &f) {
  return f.d == 1 ? t : (int)(((uint64_t)(uint32_t)t * f.m) >> 32);
}

// An axis' length, its radices, before each the product of those done, and the
// divisions by r (of pass 0, by n / r)
struct FftAxis {
  int n, npass;
  int r[kMaxPasses];
  FastDiv ns[kMaxPasses], rd[kMaxPasses];
};

// 0: powers of 2 only, 1: also 3 and 5, 2: any
inline int radix_kind(const FftAxis &a) {
  int kind = 0;
  for (int p = 0; p < a.npass; p++)
    kind = a.r[p] > 5 && a.r[p] != 8 ? 2 : (a.r[p] == 3 || a.r[p] == 5) && kind == 0 ? 1 : kind;
  return kind;
}

// Splits n into radices; false if a prime factor is above 13 and `largest`
inline bool fft_axis(int n, int largest, FftAxis *a) {
  a->n = n;
  a->npass = 0;
  auto take = [&](int r) {
    while (n % r == 0 && a->npass < kMaxPasses) {
      a->ns[a->npass] = fast_div(a->n / n);
      a->rd[a->npass] = fast_div(a->npass == 0 ? a->n / r : r);
      a->r[a->npass++] = r;
      n /= r;
    }
  };
  // the large primes (an odd p without these factors is one, or a product of
  // primes that have been taken)
  for (int p = 17; p <= largest; p += 2)
    if (p % 3 && p % 5 && p % 7 && p % 11 && p % 13) take(p);
  // 16 = 4 x 4 and not 8 x 2
  if (n % 16 == 0 && n % 32 != 0) take(4);
  take(8);
  take(4);
  take(2);
  for (int p = 3; p <= 13; p += 2) take(p);
  return n == 1;
}

__host__ __device__ inline double2 cadd(double2 a, double2 b) {
  return make_double2(a.x + b.x, a.y + b.y);
}
__host__ __device__ inline double2 csub(double2 a, double2 b) {
  return make_double2(a.x - b.x, a.y - b.y);
}
__host__ __device__ inline double2 cscale(double2 a, double f) {
  return make_double2(a.x * f, a.y * f);
}
// a w, or a conj(w) for the inverse transform
template <bool INV>
__host__ __device__ inline double2 cmul(double2 a, double2 w) {
  const double wy = INV ? -w.y : w.y;
  return make_double2(a.x * w.x - a.y * wy, a.x * wy + a.y * w.x);
}
// -i a (forward), i a (inverse)
template <bool INV>
__host__ __device__ inline double2 crot(double2 a) {
  return INV ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x);
}

// cos and sin of 2 pi k / R, k = 0 .. R / 2
template <int R>
struct RootsOf;
template <>
struct RootsOf<5> {
  static constexpr double c[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410};
  static constexpr double s[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
};
template <>
struct RootsOf<7> {
  static constexpr double c[4] = {1.0, 0.6234898018587335305, -0.222520933956314404,
                                  -0.900968867902419126};
  static constexpr double s[4] = {0.0, 0.7818314824680298087, 0.9749279121818236070,
                                  0.4338837391175581204};
};
template <>
struct RootsOf<11> {
  static constexpr double c[6] = {1.0,
                                  0.8412535328311811688,
                                  0.4154150130018864255,
                                  -0.142314838273285140,
                                  -0.654860733945285064,
                                  -0.959492973614497389};
  static constexpr double s[6] = {0.0,
                                  0.5406408174555975821,
                                  0.9096319953545183714,
                                  0.9898214418809327323,
                                  0.7557495743542582837,
                                  0.2817325568414296977};
};
template <>
struct RootsOf<13> {
  static constexpr double c[7] = {1.0,
                                  0.8854560256532098959,
                                  0.5680647467311558025,
                                  0.1205366802553230533,
                                  -0.354604887042535625,
                                  -0.748510748171101098,
                                  -0.970941817426052027};
  static constexpr double s[7] = {0.0,
                                  0.4647231720437685456,
                                  0.8229838658936563945,
                                  0.9927088740980539928,
                                  0.9350162426854148234,
                                  0.6631226582407952023,
                                  0.2393156642875577671};
};

template <int R, bool INV>
__host__ __device__ inline void dft(double2 v[R]) {
  if constexpr (R == 2) {
    const double2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 3) {
    constexpr double h = 0.86602540378443864676;  // sin(2 pi / 3)
    const double2 s = cadd(v[1], v[2]), d = crot<INV>(cscale(csub(v[1], v[2]), h));
    const double2 m = make_double2(v[0].x - 0.5 * s.x, v[0].y - 0.5 * s.y);
    v[0] = cadd(v[0], s);
    v[1] = cadd(m, d);
    v[2] = csub(m, d);
  } else if constexpr (R == 4) {
    const double2 a = cadd(v[0], v[2]), b = csub(v[0], v[2]), c = cadd(v[1], v[3]),
                  d = crot<INV>(csub(v[1], v[3]));
    v[0] = cadd(a, c);
    v[1] = cadd(b, d);
    v[2] = csub(a, c);
    v[3] = csub(b, d);
  } else if constexpr (R == 5 || R == 7 || R == 11 || R == 13) {
    // by the sums a and differences b of values p and R - p
    constexpr int H = R / 2;
    double2 a[H + 1], b[H + 1];
    const double2 v0 = v[0];
#pragma unroll
    for (int p = 1; p <= H; p++) {
      a[p] = cadd(v[p], v[R - p]);
      b[p] = csub(v[p], v[R - p]);
      v[0] = cadd(v[0], a[p]);
    }
#pragma unroll
    for (int q = 1; q <= H; q++) {
      double2 m = v0, d = make_double2(0.0, 0.0);
#pragma unroll
      for (int p = 1; p <= H; p++) {
        const int k = p * q % R;  // cos(2 pi k / R), sin(2 pi k / R)
        const double c = RootsOf<R>::c[k <= H ? k : R - k],
                     s = k <= H ? RootsOf<R>::s[k] : -RootsOf<R>::s[R - k];
        m.x += c * a[p].x;
        m.y += c * a[p].y;
        d.x += s * b[p].x;
        d.y += s * b[p].y;
      }
      d = crot<INV>(d);
      v[q] = cadd(m, d);
      v[R - q] = csub(m, d);
    }
  } else {
    static_assert(R == 8, "radix");
    constexpr double h = 0.70710678118654752440;
    double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft<4, INV>(e);
    dft<4, INV>(o);
    const double2 t1 = cscale(cadd(o[1], crot<INV>(o[1])), h);
    const double2 t2 = crot<INV>(o[2]);
    const double2 t3 = cscale(csub(crot<INV>(o[3]), o[3]), h);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cadd(e[1], t1);
    v[5] = csub(e[1], t1);
    v[2] = cadd(e[2], t2);
    v[6] = csub(e[2], t2);
    v[3] = cadd(e[3], t3);
    v[7] = csub(e[3], t3);
  }
}

// the butterflies of radix R over `lines` lines of n elements
template <int R, bool INV>
__host__ __device__ inline void fft_pass(const double2 *x, double2 *y, int n, FastDiv nsd,
                                         FastDiv lines, int stride, const double2 *tw, int tid,
                                         int nt) {
  const int ns = nsd.d, nr = n / R, m = nr / ns;  // m = n / (ns R)
  for (int t = tid; t < nr * lines.d; t += nt) {
    const int j = div(t, lines), l = t - j * lines.d;
    const int b = div(j, nsd), k = j - b * ns;
    double2 v[R];
    const double2 *xi = x + j * stride + l;
#pragma unroll
    for (int p = 0; p < R; p++) v[p] = xi[p * (nr * stride)];
    if (ns > 1) {
      const double2 *w = tw + k * m;
#pragma unroll
      for (int p = 1; p < R; p++, w += k * m) v[p] = cmul<INV>(v[p], *w);
    }
    dft<R, INV>(v);
    double2 *yo = y + (j + b * ns * (R - 1)) * stride + l;
#pragma unroll
    for (int q = 0; q < R; q++) yo[q * (ns * stride)] = v[q];
  }
}

// the same for any radix r, one output at a time
template <bool INV>
__host__ __device__ inline void fft_pass_any(const double2 *x, double2 *y, int n, int r, FastDiv nsd,
                                             FastDiv rd, FastDiv lines, int stride, const double2 *tw, int tid,
                                             int nt) {
  const int ns = nsd.d, nr = n / r, m = nr / ns;
  for (int t = tid; t < n * lines.d; t += nt) {
    const int o = div(t, lines), l = t - o * lines.d;  // output element
    const int bq = div(o, nsd), k = o - bq * ns, b = div(bq, rd), q = bq - b * r;
    const int j = b * ns + k, step = k * m + q * nr;  // < n
    double2 s = x[j * stride + l];
    int e = step;
    for (int p = 1; p < r; p++) {
      s = cadd(s, cmul<INV>(x[(j + p * nr) * stride + l], tw[e]));
      e += step;
      if (e >= n) e -= n;
    }
    y[o * stride + l] = s;
  }
}

// the first pass of an odd radix r: results q and r - q of each j, from the sums
// and differences of inputs p and r - p
template <bool INV>
__host__ __device__ inline void fft_pass_first(const double2 *x, double2 *y, int n, int r,
                                               FastDiv lines, FastDiv nrd, int stride,
                                               const double2 *tw, int tid, int nt) {
  const int nr = nrd.d, h = r / 2;
  for (int t = tid; t < nr * lines.d * (h + 1); t += nt) {
    const int jq = div(t, lines), l = t - jq * lines.d;
    const int q = div(jq, nrd), j = jq - q * nr;
    const double2 *a = x + j * stride + l, *b = a + n * stride;
    const int step = q * nr, by = nr * stride;
    double2 m = *a, d = make_double2(0.0, 0.0);
    int e = 0;
    for (int p = 1; p <= h; p++) {
      a += by;
      b -= by;
      e += step;
      if (e >= n) e -= n;
      const double2 w = tw[e], u = *a, v = *b;  // (cos, -sin)
      m.x += w.x * (u.x + v.x);
      m.y += w.x * (u.y + v.y);
      d.x -= w.y * (u.x - v.x);
      d.y -= w.y * (u.y - v.y);
    }
    d = crot<INV>(d);
    double2 *o = y + j * r * stride + l;
    o[q * stride] = cadd(m, d);
    if (q > 0) o[(r - q) * stride] = csub(m, d);
  }
}

// a value that is the same for the whole wave, as a scalar
__host__ __device__ inline int uniform(int v) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_readfirstlane(v);
#else
  return v;
#endif
}
__host__ __device__ inline FastDiv uniform(const FastDiv &f) {
  return FastDiv{(uint32_t)uniform((int)f.m), uniform(f.d)};
}

// One pass of axis a: x -> y.  KIND is the largest kind (radix_kind) of its
// axes: a kernel holds the code of no other radix (16^3 cells' solve takes 1.3 us
// longer with all of them, which are then fetched past).
template <bool INV, int KIND>
__host__ __device__ inline void fft_pass_of(const FftAxis &a, int pass, const double2 *x,
                                            double2 *y, FastDiv lines, int stride,
                                            const double2 *tw, int tid, int nt) {
  const FastDiv ns = uniform(a.ns[pass]);
  const int r = uniform(a.r[pass]), n = uniform(a.n);
  auto go = [&](auto radix) {
    fft_pass<decltype(radix)::value, INV>(x, y, n, ns, lines, stride, tw, tid, nt);
  };
  if (r == 8) return go(std::integral_constant<int, 8>());
  if (r == 4) return go(std::integral_constant<int, 4>());
  if (KIND == 0 || r == 2) return go(std::integral_constant<int, 2>());
  if constexpr (KIND >= 1) {
    if (r == 3) return go(std::integral_constant<int, 3>());
    if (KIND == 1 || r == 5) return go(std::integral_constant<int, 5>());
  }
  if constexpr (KIND >= 2) {
    if (r == 7) return go(std::integral_constant<int, 7>());
    if (r == 11) return go(std::integral_constant<int, 11>());
    if (r == 13) return go(std::integral_constant<int, 13>());
    if (pass == 0)
      fft_pass_first<INV>(x, y, n, r, lines, uniform(a.rd[0]), stride, tw, tid, nt);
    else
      fft_pass_any<INV>(x, y, n, r, ns, uniform(a.rd[pass]), lines, stride, tw, tid, nt);
  }
}

// Two real lines a, b went through one transform as a + i b.  Splits the result
// z[k * stride + p] (pair p of np) into the half spectra y[line * hx + k].
__host__ __device__ inline void split_pairs(const double2 *z, int stride, double2 *y, int nx, int ny,
                                            FastDiv np, int tid, int nt) {
  const int hx = nx / 2 + 1;
  for (int t = tid; t < hx * np.d; t += nt) {
    const int k = div(t, np), p = t - k * np.d;
    const double2 u = z[k * stride + p], w = z[(k == 0 ? 0 : nx - k) * stride + p];
    if (2 * p < ny) y[2 * p * hx + k] = make_double2(0.5 * (u.x + w.x), 0.5 * (u.y - w.y));
    if (2 * p + 1 < ny)
      y[(2 * p + 1) * hx + k] = make_double2(0.5 * (u.y + w.y), 0.5 * (w.x - u.x));
  }
}

// The inverse: the whole spectra of a + i b from the half spectra of a and b
// (whose zero and middle modes are real)
__host__ __device__ inline void join_pairs(const double2 *y, double2 *z, int stride, int nx, int ny,
                                           FastDiv np, int tid, int nt) {
  const int hx = nx / 2 + 1;
  for (int t = tid; t < hx * np.d; t += nt) {
    const int k = div(t, np), p = t - k * np.d;
    double2 a = 2 * p < ny ? y[2 * p * hx + k] : make_double2(0.0, 0.0);
    double2 b = 2 * p + 1 < ny ? y[(2 * p + 1) * hx + k] : make_double2(0.0, 0.0);
    const bool real = k == 0 || 2 * k == nx;
    if (real) a.y = b.y = 0.0;
    z[k * stride + p] = make_double2(a.x - b.y, a.y + b.x);
    if (!real) z[(nx - k) * stride + p] = make_double2(a.x + b.y, b.x - a.y);
  }
}

}  // namespace emg
#endif
