// phases.h -- device helpers shared by the phase kernels (p2m.hip, l2p.hip,
// translate.hip, m2l.hip, p2p.hip): solid harmonics, Bessel factors, box
// centres, MFMA wrappers and the dispatch over expansion orders.
#pragma once

#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "engine.h"
#include "m2l.h"
#include "mfma.h"
#include "tree_util.h"

namespace fmmx {

namespace {

// ---------------------------------------------------------------------
// Coefficients of the solid-harmonic recurrences, S_n^m = rho^n fac P_n^m e^{im beta}
// with fac = sqrt((n-m)!/(n+m)!) and the Condon-Shortley phase
// (kernel/multipole.cxx:7-35):
//   S_m^m     = -a_m (x+iy) S_{m-1}^{m-1},      a_m = sqrt((2m-1)/(2m))
//   S_{m+1}^m = b_m z S_m^m,                    b_m = sqrt(2m+1)
//   S_{n+1}^m = c_nm z S_n^m - d_nm r^2 S_{n-1}^m
// and of their derivatives (d/dx + i d/dy) S_n^m = gp_nm S_{n-1}^{m+1},
// (d/dx - i d/dy) S_n^m = -gm_nm S_{n-1}^{m-1}, d/dz S_n^m = gz_nm S_{n-1}^m.
constexpr double csqrt(double x) {
  if (x <= 0) return 0;
  double r = x > 1 ? x : 1;
  for (int i = 0; i < 200; i++) r = 0.5 * (r + x / r);
  return r;
}
struct HarmCoef {
  double a[MAXP + 2], b[MAXP + 2], c[MAXP + 2][MAXP + 2], d[MAXP + 2][MAXP + 2];
  double gp[MAXP + 2][MAXP + 2], gm[MAXP + 2][MAXP + 2], gz[MAXP + 2][MAXP + 2];
};
constexpr HarmCoef make_coef() {
  HarmCoef h{};
  for (int m = 0; m <= MAXP + 1; m++) {
    h.a[m] = m > 0 ? csqrt((2.0 * m - 1) / (2.0 * m)) : 0;
    h.b[m] = csqrt(2.0 * m + 1);
  }
  for (int n = 0; n <= MAXP + 1; n++)
    for (int m = 0; m <= MAXP + 1; m++) {
      double den = (double)(n + 1 - m) * (n + 1 + m);
      h.c[n][m] = den > 0 ? (2.0 * n + 1) / csqrt(den) : 0;
      h.d[n][m] = den > 0 ? csqrt((double)(n - m) * (n + m) / den) : 0;
      h.gp[n][m] = (n - m) * (n - m - 1) > 0 ? csqrt((double)(n - m) * (n - m - 1)) : 0;
      h.gm[n][m] = (n + m) * (n + m - 1) > 0 ? csqrt((double)(n + m) * (n + m - 1)) : 0;
      h.gz[n][m] = (n - m) * (n + m) > 0 ? csqrt((double)(n - m) * (n + m)) : 0;
    }
  return h;
}
__constant__ HarmCoef c_hc = make_coef();

__host__ __device__ constexpr int sl(int n, int m) { return n * (n + 1) / 2 + m; }
// the same coefficients rounded to float once, read by uniform (scalar) loads
struct HarmCoefF {
  float a[MAXP + 2], b[MAXP + 2], c[MAXP + 2][MAXP + 2], d[MAXP + 2][MAXP + 2];
};
constexpr HarmCoefF make_coef_f() {
  const HarmCoef h = make_coef();
  HarmCoefF f{};
  for (int m = 0; m <= MAXP + 1; m++) {
    f.a[m] = (float)h.a[m];
    f.b[m] = (float)h.b[m];
    for (int n = 0; n <= MAXP + 1; n++) {
      f.c[n][m] = (float)h.c[n][m];
      f.d[n][m] = (float)h.d[n][m];
    }
  }
  return f;
}
__constant__ HarmCoefF c_hcf = make_coef_f();
template <typename T>
struct HC {
  static __device__ __forceinline__ T a(int m) { return T(c_hc.a[m]); }
  static __device__ __forceinline__ T b(int m) { return T(c_hc.b[m]); }
  static __device__ __forceinline__ T c(int n, int m) { return T(c_hc.c[n][m]); }
  static __device__ __forceinline__ T d(int n, int m) { return T(c_hc.d[n][m]); }
};
template <>
struct HC<float> {
  static __device__ __forceinline__ float a(int m) { return c_hcf.a[m]; }
  static __device__ __forceinline__ float b(int m) { return c_hcf.b[m]; }
  static __device__ __forceinline__ float c(int n, int m) { return c_hcf.c[n][m]; }
  static __device__ __forceinline__ float d(int n, int m) { return c_hcf.d[n][m]; }
};



template <int P, typename T>
__device__ __forceinline__ void solid_harmonics(T x, T y, T z, T* Sr, T* Si) {
  const T r2 = x * x + y * y + z * z;
  Sr[0] = T(1);
  Si[0] = T(0);
#pragma unroll
  for (int m = 0; m < P; m++) {
    if (m > 0) {
      const T a = -T(c_hc.a[m]);
      const int pm = sl(m - 1, m - 1);
      Sr[sl(m, m)] = a * (x * Sr[pm] - y * Si[pm]);
      Si[sl(m, m)] = a * (x * Si[pm] + y * Sr[pm]);
    }
    if (m + 1 < P) {
      const T b = T(c_hc.b[m]) * z;
      Sr[sl(m + 1, m)] = b * Sr[sl(m, m)];
      Si[sl(m + 1, m)] = b * Si[sl(m, m)];
    }
#pragma unroll
    for (int n = m + 1; n + 1 < P; n++) {
      const T c = T(c_hc.c[n][m]) * z, d = T(c_hc.d[n][m]) * r2;
      Sr[sl(n + 1, m)] = c * Sr[sl(n, m)] - d * Sr[sl(n - 1, m)];
      Si[sl(n + 1, m)] = c * Si[sl(n, m)] - d * Si[sl(n - 1, m)];
    }
  }
}

// Gradient of S_n^m (n >= 1) in terms of degree n-1 values:
// dS/dx = (Ap + Am)/2, dS/dy = -i (Ap - Am)/2, dS/dz = gz S_{n-1}^m
template <int P, typename T>
__device__ __forceinline__ void harm_grad(const T* Sr, const T* Si, int n, int m, T& pr, T& pi, T& mr, T& mi,
                                          T& zr, T& zi) {
  pr = pi = mr = mi = zr = zi = T(0);
  if (m + 1 <= n - 1) {
    const T g = T(c_hc.gp[n][m]);
    pr = g * Sr[sl(n - 1, m + 1)];
    pi = g * Si[sl(n - 1, m + 1)];
  }
  if (m >= 1) {
    const T g = -T(c_hc.gm[n][m]);
    mr = g * Sr[sl(n - 1, m - 1)];
    mi = g * Si[sl(n - 1, m - 1)];
  } else if (n >= 2) {
    const T g = T(c_hc.gp[n][0]);  // m = 0: conj(S_{n-1}^1) term
    mr = g * Sr[sl(n - 1, 1)];
    mi = -g * Si[sl(n - 1, 1)];
  }
  if (m <= n - 1) {
    const T g = T(c_hc.gz[n][m]);
    zr = g * Sr[sl(n - 1, m)];
    zi = g * Si[sl(n - 1, m)];
  }
}

// Evaluation point of an expansion in units of the box size.  REF: the
// reference's angles (kernel/G_p2m.cxx:31-41) with eps added to the radius
// and float pi in the azimuth branches; the harmonics at these angles equal
// the solid harmonics at the point below.
__device__ __forceinline__ void eff_point(int conv, double dx, double dy, double dz, double rbinv, double& ux,
                                          double& uy, double& uz) {
  if (conv == FMMX_CONV_EXACT) {
    ux = dx * rbinv;
    uy = dy * rbinv;
    uz = dz * rbinv;
    return;
  }
  const double eps = (double)EPSF, pif = (double)PIF;
  double rh = sqrt(dx * dx + dy * dy + dz * dz) + eps;
  double ca = cos(acos(dz / rh));
  double sa = sqrt((1 - ca) * (1 + ca));
  double be;
  if (fabs(dx) + fabs(dy) < eps) be = 0;
  else if (fabs(dx) < eps) be = dy / fabs(dy) * pif * 0.5;
  else if (dx > 0) be = atan(dy / dx);
  else be = atan(dy / dx) + pif;
  double sb, cb;
  sincos(be, &sb, &cb);
  ux = rh * sa * cb * rbinv;
  uy = rh * sa * sb * rbinv;
  uz = rh * ca * rbinv;
}

// i~_n(x) = i_n(x) / x^n for n = 0..N (modified spherical Bessel function
// of the first kind over x^n): power series for N+1 and N, then the stable
// backward recurrence i~_{n-1} = (2n+1) i~_n + x^2 i~_{n+1}
template <int N>
__device__ inline void ibar_dev(double x, double* out) {
  const double h = 0.5 * x * x;
  double top[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int n = N + 1 - u;
    double df = 1;
    for (int k = 3; k <= 2 * n + 1; k += 2) df *= k;
    double t = 1.0 / df, sum = t;
    for (int k = 1; k < 400; k++) {
      t *= h / (k * (2.0 * n + 2.0 * k + 1.0));
      sum += t;
      if (t < 1e-18 * sum) break;
    }
    top[u] = sum;
  }
  double a = top[0], b = top[1];
  out[N] = b;
#pragma unroll
  for (int n = N; n >= 1; n--) {
    const double c = (2 * n + 1) * b + x * x * a;
    a = b;
    b = c;
    out[n - 1] = c;
  }
}

// j^_n(x) = (2n+1)!! j_n(x) / x^n for n = 0..N (spherical Bessel function of
// the first kind, scaled to 1 at x = 0): power series for N+1 and N, then
// the stable backward recurrence j^_{n-1} = j^_n - x^2 j^_{n+1}/((2n+1)(2n+3))
template <int N>
__device__ inline void jhat_dev(double x, double* out) {
  const double h = -0.5 * x * x;
  double top[2];
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int n = N + 1 - u;
    double t = 1, sum = 1, tmax = 1;
    for (int k = 1; k < 400; k++) {
      t *= h / (k * (2.0 * n + 2.0 * k + 1.0));
      sum += t;
      tmax = fmax(tmax, fabs(t));
      if (fabs(t) < 1e-18 * tmax) break;
    }
    top[u] = sum;
  }
  double a = top[0], b = top[1];
  out[N] = b;
#pragma unroll
  for (int n = N; n >= 1; n--) {
    const double c = b - x * x * a / ((2.0 * n + 1.0) * (2.0 * n + 3.0));
    a = b;
    b = c;
    out[n - 1] = c;
  }
}

__device__ __forceinline__ void box_center(uint32_t key, int lev, double xmin, double ymin, double zmin, double rb,
                                           double& cx, double& cy, double& cz) {
  int ix, iy, iz;
  morton_decode(key, lev, ix, iy, iz);
  cx = xmin + (ix + 0.5) * rb;
  cy = ymin + (iy + 0.5) * rb;
  cz = zmin + (iz + 0.5) * rb;
}

template <typename T>
__global__ void k_m2l_reduce(long n, int nsplit, const T* __restrict__ part, T* __restrict__ L, int init) {
  const long e = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  T s = init ? T(0) : L[e];
  for (int k = 0; k < nsplit; k++) s += part[(size_t)k * n + e];
  L[e] = s;
}

template <class T>
struct tag {
  using type = T;
};

template <typename F>
int dispatch_p(int p, F&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(2) FMMX_CASE(3) FMMX_CASE(4) FMMX_CASE(5) FMMX_CASE(6) FMMX_CASE(7) FMMX_CASE(8) FMMX_CASE(9)
    FMMX_CASE(10) FMMX_CASE(11) FMMX_CASE(12)
#undef FMMX_CASE
  }
  return fail(FMMX_EUNSUPPORTED, "unsupported p");
}

// the orders the Helmholtz kernels are built for
template <typename F>
int dispatch_hp(int p, F&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(4) FMMX_CASE(6) FMMX_CASE(8) FMMX_CASE(10) FMMX_CASE(12)
#undef FMMX_CASE
  }
  return fail(FMMX_EUNSUPPORTED, "Helmholtz needs p in {4, 6, 8, 10, 12}");
}

// the order above P_ALL: FP64 and the EXACT convention (checked when the
// handle is created), on the vector-unit kernels
template <typename F>
int dispatch_hi(int p, F&& f) {
  if (p == P_HI) return f(std::integral_constant<int, P_HI>{});
  return fail(FMMX_EUNSUPPORTED, "unsupported p");
}

}  // namespace

}  // namespace fmmx
