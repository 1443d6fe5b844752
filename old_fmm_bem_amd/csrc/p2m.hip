// p2m.hip -- P2M (kernel/G_p2m.cxx, Gn_p2m.cxx) for CDNA4 (gfx950), wave64: one
// wave per leaf box (two leaves per wave when small); solid harmonics from a
// Cartesian recurrence (no acos/atan per term).
#include "phases.h"

namespace fmmx {

namespace {

// ---------------------------------------------------------------------
// P2M: one wave per source leaf box
//   YK 1: Yukawa multipoles, M~_n^m = sum q i~_n(lambda rho)/i~_n(lambda rb)
//       (rho/rb)^n conj(Y_n^m): the Laplace harmonics times a radial weight
//       per degree (lrb = lambda rb)
//   YK 2: Helmholtz multipoles, M_n^m = sum q j^_n(k rho) (rho/rb)^n
//       conj(Y_n^m) (lrb = k rb), of the real charges q and the imaginary ones
//       q2 (VS behind).  Both parts in one pass: the Bessel series in FP64 and
//       the harmonics are most of the work (sphere of 1M points, p = 12, beside the near
//       field: 0.96 ms as a pass per part, 0.86 ms here)
//   Box b's multipole starts at M + b * mstride + moff.
template <int P, typename T, int YK = 0, int HALF = 0, int CONV = -1, int GN = -1>
__global__ __launch_bounds__(64) void k_p2m(int nb, const uint32_t* __restrict__ bkey, const int* __restrict__ bfirst,
                                            const int* __restrict__ blast, const float* __restrict__ x,
                                            const float* __restrict__ y, const float* __restrict__ z,
                                            const float* __restrict__ nx, const float* __restrict__ ny,
                                            const float* __restrict__ nz, const float* __restrict__ q, int gn,
                                            int conv, int lev, double xmin, double ymin, double zmin, double rb,
                                            const double* __restrict__ corr, T* __restrict__ M, double lrb,
                                            int mstride, int moff, const float* __restrict__ q2) {
  // HALF: two leaves per wave, rows 0-31 for the first and 32-63 for the
  // second, for leaves of at most about 32 particles
  constexpr int NR = P * (P + 1) / 2, P2 = P * P, NL = HALF ? 2 : 1, STEP = 64 / NL;
  constexpr int NC = (NL * P2 + 63) / 64, PARTS = YK == 2 ? 2 : 1;
  __shared__ T red[64][P2 + 1];
  const int lane = threadIdx.x, h = HALF ? lane >> 5 : 0, sub = HALF ? lane & 31 : lane;
  const int b = HALF ? 2 * (int)blockIdx.x + h : (int)blockIdx.x;
  const bool valid = b < nb;
  if (!HALF && !valid) return;
  double cx = 0, cy = 0, cz = 0;
  if (valid) box_center(bkey[b], lev, xmin, ymin, zmin, rb, cx, cy, cz);
  const double rbinv = 1.0 / rb;
  T acc[PARTS][NC];
#pragma unroll
  for (int t = 0; t < PARTS; t++)
#pragma unroll
    for (int c = 0; c < NC; c++) acc[t][c] = T(0);
  // column sums: entry idx = (leaf of the wave, column) over that leaf's rows
  auto sums = [&](int t) __attribute__((always_inline)) {
    __syncthreads();
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int idx = lane + 64 * c, hh = idx / P2, col = idx % P2;
      if (hh < NL) {
        T s = T(0);
        for (int r = 0; r < STEP; r++) s += red[hh * STEP + r][col];
        acc[t][c] += s;
      }
    }
    __syncthreads();
  };
  const int i0 = valid ? bfirst[b] : 0, i1 = valid ? blast[b] : -1;
  for (int base = 0;; base += STEP) {
    if (__ballot(i0 + base <= i1) == 0) break;  // one wave per block: uniform
    const int i = i0 + base + sub;
    T* row = red[lane];
    if constexpr (YK == 2) {
      double ux = 0, uy = 0, uz = 0, jx[P];
      if (i <= i1)
        eff_point(CONV >= 0 ? CONV : conv, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
      T Sr[NR], Si[NR];
      solid_harmonics<P, T>(T(ux), T(uy), T(uz), Sr, Si);
      jhat_dev<P - 1>(lrb * sqrt(ux * ux + uy * uy + uz * uz), jx);
#pragma unroll
      for (int t = 0; t < PARTS; t++) {
        const double qd = i <= i1 ? (double)(t ? q2 : q)[i] : 0.0;
#pragma unroll
        for (int n = 0; n < P; n++) {
          const T w = T(qd * jx[n]);
#pragma unroll
          for (int m = 0; m <= n; m++) {
            row[sl(n, m)] = w * Sr[sl(n, m)];
            if (m > 0) row[NR + n * (n - 1) / 2 + m - 1] = -w * Si[sl(n, m)];
          }
        }
        sums(t);
      }
      continue;
    }
    if (YK == 0 && CONV == FMMX_CONV_EXACT && GN == 0 && i <= i1) {
      // charges in the EXACT convention (unit table ratios): the harmonics
      // column by column straight into the LDS row; the unrolled recurrence
      // uses literal coefficients and keeps only its state live
      double ux, uy, uz;
      eff_point(FMMX_CONV_EXACT, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
      const T tx = T(ux), ty = T(uy), tz = T(uz), r2 = tx * tx + ty * ty + tz * tz, qi = T(q[i]);
      constexpr HarmCoef hc = make_coef();
      auto put = [&](int n, int m, T sr, T si) {
        row[sl(n, m)] = qi * sr;
        if (m > 0) row[NR + n * (n - 1) / 2 + m - 1] = -qi * si;
      };
      T dr = T(1), di = T(0);
#pragma unroll
      for (int m = 0; m < P; m++) {
        if (m > 0) {
          const T a = -T(hc.a[m]), nr = a * (tx * dr - ty * di), ni = a * (tx * di + ty * dr);
          dr = nr;
          di = ni;
        }
        put(m, m, dr, di);
        if (m + 1 < P) {
          const T bz = T(hc.b[m]) * tz;
          T pr = dr, pi = di, sr = bz * dr, si = bz * di;
          put(m + 1, m, sr, si);
#pragma unroll
          for (int n = m + 2; n < P; n++) {
            const T cz = T(hc.c[n - 1][m]) * tz, d = T(hc.d[n - 1][m]) * r2;
            const T nr = cz * sr - d * pr, ni = cz * si - d * pi;
            pr = sr;
            pi = si;
            sr = nr;
            si = ni;
            put(n, m, sr, si);
          }
        }
      }
    } else if (i <= i1) {
      const int cv = CONV >= 0 ? CONV : conv;
      const int gnv = GN >= 0 ? GN : gn;
      double ux, uy, uz;
      eff_point(cv, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
      T Sr[NR], Si[NR];
      solid_harmonics<P, T>(T(ux), T(uy), T(uz), Sr, Si);
      if (YK) {
        double ib0[P], ibx[P];
        const double lr = lrb * sqrt(ux * ux + uy * uy + uz * uz);
        ibar_dev<P - 1>(lrb, ib0);
        ibar_dev<P - 1>(lr, ibx);
        const double qd = (double)q[i];
#pragma unroll
        for (int n = 0; n < P; n++) {
          const T w = T(qd * ibx[n] / ib0[n]);
#pragma unroll
          for (int m = 0; m <= n; m++) {
            row[sl(n, m)] = w * Sr[sl(n, m)];
            if (m > 0) row[NR + n * (n - 1) / 2 + m - 1] = -w * Si[sl(n, m)];
          }
        }
      } else if (!gnv) {
        const T qi = T(q[i]);
#pragma unroll
        for (int n = 0; n < P; n++)
#pragma unroll
          for (int m = 0; m <= n; m++) {
            const T w = qi * T(corr[sl(n, m)]);
            row[sl(n, m)] = w * Sr[sl(n, m)];
            if (m > 0) row[NR + n * (n - 1) / 2 + m - 1] = -w * Si[sl(n, m)];
          }
      } else {
        // dipole q*n (the float product vj*gxj of kernel/Gn_p2m.cxx:113)
        const T qx = T(q[i] * nx[i]), qy = T(q[i] * ny[i]), qz = T(q[i] * nz[i]);
        row[0] = T(0);
#pragma unroll
        for (int n = 1; n < P; n++)
#pragma unroll
          for (int m = 0; m <= n; m++) {
            T pr, pi, mr, mi, zr, zi;
            harm_grad<P, T>(Sr, Si, n, m, pr, pi, mr, mi, zr, zi);
            // n . grad S = qx (Ap+Am)/2 + qy (-i)(Ap-Am)/2 + qz dS/dz
            const T dr = T(0.5) * qx * (pr + mr) + T(0.5) * qy * (pi - mi) + qz * zr;
            const T di = T(0.5) * qx * (pi + mi) - T(0.5) * qy * (pr - mr) + qz * zi;
            const T w = T(corr[sl(n, m)] * rbinv);
            row[sl(n, m)] = w * dr;
            if (m > 0) row[NR + n * (n - 1) / 2 + m - 1] = -w * di;
          }
      }
    } else {
#pragma unroll
      for (int c = 0; c < P2; c++) row[c] = T(0);
    }
    sums(0);
  }
  using ML = MLayout<P>;
  const int b0 = HALF ? 2 * (int)blockIdx.x : (int)blockIdx.x;
#pragma unroll
  for (int t = 0; t < PARTS; t++)
#pragma unroll
    for (int c = 0; c < NC; c++) {
      const int idx = lane + 64 * c, hh = idx / P2, col = idx % P2;
      if (hh < NL && b0 + hh < nb) M[(size_t)(b0 + hh) * mstride + moff + t * ML::VS + ML::at(col)] = acc[t][c];
    }
  // zero the padding slots (M2M applies its operator to whole stored vectors)
  for (int c2 = lane; c2 < NL * ML::VS; c2 += 64) {
    const int hh = c2 / ML::VS, c = c2 % ML::VS;
    if (b0 + hh < nb && (c % ML::KSP >= ML::KS || (c / ML::KSP) * ML::KS + c % ML::KSP >= P2))
#pragma unroll
      for (int t = 0; t < PARTS; t++) M[(size_t)(b0 + hh) * mstride + moff + t * ML::VS + c] = T(0);
  }
}

// P2M above order 12 (FP64, EXACT convention): a 64 x P^2 table of particle
// terms (166 KB at P = 18) no longer fits LDS, so each lane keeps its
// particle's harmonics in registers (spilled as the compiler needs) and the
// table goes through LDS 64 columns at a time, each column summed by one lane
// in fixed row order (deterministic).  YK 1: Yukawa weights as k_p2m;
// GN 1: the dipole form of k_p2m (Gnj).
template <int P, int YK, int GN>
__global__ __launch_bounds__(64) void k_p2m_hi(int nb, const uint32_t* __restrict__ bkey,
                                               const int* __restrict__ bfirst, const int* __restrict__ blast,
                                               const float* __restrict__ x, const float* __restrict__ y,
                                               const float* __restrict__ z, const float* __restrict__ nx,
                                               const float* __restrict__ ny, const float* __restrict__ nz,
                                               const float* __restrict__ q, int lev, double xmin, double ymin,
                                               double zmin, double rb, double* __restrict__ M, double lrb) {
  constexpr int NR = P * (P + 1) / 2, P2 = P * P, CH = 64, NC = (P2 + CH - 1) / CH;
  __shared__ double red[64][CH + 1];
  const int lane = threadIdx.x, b = blockIdx.x;
  if (b >= nb) return;  // one wave per block: uniform
  double cx, cy, cz;
  box_center(bkey[b], lev, xmin, ymin, zmin, rb, cx, cy, cz);
  const double rbinv = 1.0 / rb;
  double acc[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) acc[c] = 0;
  double ib0[P];
  if (YK) ibar_dev<P - 1>(lrb, ib0);
  const int i0 = bfirst[b], i1 = blast[b];
  for (int base = i0; base <= i1; base += 64) {
    const int i = base + lane;
    const bool on = i <= i1;
    double Sr[NR], Si[NR], w[P];
    const double ux = on ? ((double)x[i] - cx) * rbinv : 0, uy = on ? ((double)y[i] - cy) * rbinv : 0,
                 uz = on ? ((double)z[i] - cz) * rbinv : 0;
    solid_harmonics<P, double>(ux, uy, uz, Sr, Si);
    const double qi = on ? (double)q[i] : 0;
    if (YK) {
      double ibx[P];
      ibar_dev<P - 1>(lrb * sqrt(ux * ux + uy * uy + uz * uz), ibx);
#pragma unroll
      for (int n = 0; n < P; n++) w[n] = qi * ibx[n] / ib0[n];
    } else {
#pragma unroll
      for (int n = 0; n < P; n++) w[n] = GN ? rbinv : qi;
    }
    // dipole q*n: the float product vj*gxj of kernel/Gn_p2m.cxx:113, as k_p2m
    const double qx = GN && on ? (double)(q[i] * nx[i]) : 0, qy = GN && on ? (double)(q[i] * ny[i]) : 0,
                 qz = GN && on ? (double)(q[i] * nz[i]) : 0;
    // column col of this particle's row: Re slots sl(n, m), then Im slots
    auto term = [&](int n, int m, bool im) -> double {
      if (GN) {
        if (n == 0) return 0;
        double pr, pi, mr, mi, zr, zi;
        harm_grad<P, double>(Sr, Si, n, m, pr, pi, mr, mi, zr, zi);
        if (!im) return w[n] * (0.5 * qx * (pr + mr) + 0.5 * qy * (pi - mi) + qz * zr);
        return -w[n] * (0.5 * qx * (pi + mi) - 0.5 * qy * (pr - mr) + qz * zi);
      }
      return im ? -w[n] * Si[sl(n, m)] : w[n] * Sr[sl(n, m)];
    };
#pragma unroll
    for (int c = 0; c < NC; c++) {
#pragma unroll
      for (int n = 0; n < P; n++)
#pragma unroll
        for (int m = 0; m <= n; m++) {
          const int cr = sl(n, m), cim = NR + n * (n - 1) / 2 + m - 1;
          if (cr >= c * CH && cr < (c + 1) * CH) red[lane][cr - c * CH] = term(n, m, false);
          if (m > 0 && cim >= c * CH && cim < (c + 1) * CH) red[lane][cim - c * CH] = term(n, m, true);
        }
      __syncthreads();
      if (c * CH + lane < P2) {
        double s = 0;
        for (int r = 0; r < 64; r++) s += red[r][lane];
        acc[c] += s;
      }
      __syncthreads();
    }
  }
  using ML = MLayout<P>;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    const int col = c * CH + lane;
    if (col < P2) M[(size_t)b * ML::VS + ML::at(col)] = acc[c];
  }
  for (int c = lane; c < ML::VS; c += 64)
    if (c % ML::KSP >= ML::KS || (c / ML::KSP) * ML::KS + c % ML::KSP >= P2) M[(size_t)b * ML::VS + c] = 0;
}

// P2M of charges in the EXACT convention, FP32 (the mixed engine's G, Gni):
// each lane's particle terms stay in registers and the per-leaf column sums
// go through LDS in chunks of CH columns, so a workgroup holds 8-17 KB of
// LDS instead of a whole 64 x P^2 table (four to eight times the
// workgroups per CU of k_p2m).  Same leaves-per-wave forms as k_p2m.
template <int P, int HALF>
__global__ __launch_bounds__(64) void k_p2m_exact(int nb, const uint32_t* __restrict__ bkey,
                                                  const int* __restrict__ bfirst, const int* __restrict__ blast,
                                                  const float* __restrict__ x, const float* __restrict__ y,
                                                  const float* __restrict__ z, const float* __restrict__ q, int lev,
                                                  double xmin, double ymin, double zmin, double rb,
                                                  float* __restrict__ M, int mstride, int moff) {
  constexpr int NR = P * (P + 1) / 2, P2 = P * P, NL = HALF ? 2 : 1, STEP = 64 / NL;
  constexpr int CH = 64 / NL, NQ = (P2 + CH - 1) / CH;
  __shared__ float red[64][CH + 1];
  const int lane = threadIdx.x, h = HALF ? lane >> 5 : 0, sub = HALF ? lane & 31 : lane;
  const int b = HALF ? 2 * (int)blockIdx.x + h : (int)blockIdx.x;
  const bool valid = b < nb;
  if (!HALF && !valid) return;
  double cx = 0, cy = 0, cz = 0;
  if (valid) box_center(bkey[b], lev, xmin, ymin, zmin, rb, cx, cy, cz);
  const double rbinv = 1.0 / rb;
  float acc[NQ];
#pragma unroll
  for (int k = 0; k < NQ; k++) acc[k] = 0.f;
  // column sums: lane -> (leaf cl, column cc of the chunk)
  const int cl = lane / CH, cc = lane % CH;
  const int i0 = valid ? bfirst[b] : 0, i1 = valid ? blast[b] : -1;
  constexpr HarmCoef hc = make_coef();
  for (int base = 0;; base += STEP) {
    if (__ballot(i0 + base <= i1) == 0) break;  // one wave per block: uniform
    const int i = i0 + base + sub;
    float v[P2];
#pragma unroll
    for (int c = 0; c < P2; c++) v[c] = 0.f;
    if (i <= i1) {
      double ux, uy, uz;
      eff_point(FMMX_CONV_EXACT, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
      const float tx = (float)ux, ty = (float)uy, tz = (float)uz, r2 = tx * tx + ty * ty + tz * tz, qi = q[i];
      auto put = [&](int n, int m, float sr, float si) {
        v[sl(n, m)] = qi * sr;
        if (m > 0) v[NR + n * (n - 1) / 2 + m - 1] = -qi * si;
      };
      float dr = 1.f, di = 0.f;
#pragma unroll
      for (int m = 0; m < P; m++) {
        if (m > 0) {
          const float a = -(float)hc.a[m], nr = a * (tx * dr - ty * di), ni = a * (tx * di + ty * dr);
          dr = nr;
          di = ni;
        }
        put(m, m, dr, di);
        if (m + 1 < P) {
          const float bz = (float)hc.b[m] * tz;
          float pr = dr, pi = di, sr = bz * dr, si = bz * di;
          put(m + 1, m, sr, si);
#pragma unroll
          for (int n = m + 2; n < P; n++) {
            const float cz = (float)hc.c[n - 1][m] * tz, d = (float)hc.d[n - 1][m] * r2;
            const float nr = cz * sr - d * pr, ni = cz * si - d * pi;
            pr = sr;
            pi = si;
            sr = nr;
            si = ni;
            put(n, m, sr, si);
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NQ; k++) {
#pragma unroll
      for (int c = 0; c < CH; c++) red[lane][c] = k * CH + c < P2 ? v[k * CH + c] : 0.f;
      __syncthreads();
      float s0 = 0.f, s1 = 0.f;
#pragma unroll 8
      for (int r = 0; r < STEP; r += 2) {
        s0 += red[cl * STEP + r][cc];
        s1 += red[cl * STEP + r + 1][cc];
      }
      acc[k] += s0 + s1;
      __syncthreads();
    }
  }
  using ML = MLayout<P>;
  const int b0 = HALF ? 2 * (int)blockIdx.x : (int)blockIdx.x;
  if (b0 + cl < nb) {
#pragma unroll
    for (int k = 0; k < NQ; k++) {
      const int col = k * CH + cc;
      if (col < P2) M[(size_t)(b0 + cl) * mstride + moff + ML::at(col)] = acc[k];
    }
  }
  // zero the padding slots (M2M applies its operator to whole stored vectors)
  for (int c2 = lane; c2 < NL * ML::VS; c2 += 64) {
    const int hh = c2 / ML::VS, c = c2 % ML::VS;
    if (b0 + hh < nb && (c % ML::KSP >= ML::KS || (c / ML::KSP) * ML::KS + c % ML::KSP >= P2))
      M[(size_t)(b0 + hh) * mstride + moff + c] = 0.f;
  }
}

}  // namespace

int Engine::run_p2m(int neq) {
  const int nb = sj.nb[lmax];
  if (nb == 0) return FMMX_OK;
  const double* corr = corr_d.as<double>();
  if (p > P_ALL) {
    return dispatch_hi(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value;
#define FMMX_P2M_HI(YK_, GN_)                                                                                      \
  k_p2m_hi<P, YK_, GN_><<<nb, 64, 0, stream>>>(nb, sj.bkey[lmax].as<uint32_t>(), sj.bfirst[lmax].as<int>(),        \
                                               sj.blast.as<int>(), sj.x.as<float>(), sj.y.as<float>(),             \
                                               sj.z.as<float>(), sj.nx.as<float>(), sj.ny.as<float>(),             \
                                               sj.nz.as<float>(), qs.as<float>(), lmax, xmin, ymin, zmin, rb(lmax), \
                                               mexp[lmax].as<double>(), lam * rb(lmax))
      if (yk) FMMX_P2M_HI(1, 0);
      else if (neq == FMMX_GNJ) FMMX_P2M_HI(0, 1);
      else FMMX_P2M_HI(0, 0);
#undef FMMX_P2M_HI
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  return dispatch_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    const double lrb = (hh ? hk : lam) * rb(lmax);
    // two leaves per wave when leaves hold at most about 32 particles
    const bool half = (double)sj.n / nb <= 32.0;
#define FMMX_P2M_HC(T_, YK_, H_, C_, G_, Q_, STRIDE_, OFF_)                                                       \
  k_p2m<P, T_, YK_, H_, C_, G_><<<H_ ? (nb + 1) / 2 : nb, 64, 0, stream>>>(                                       \
      nb, sj.bkey[lmax].as<uint32_t>(), sj.bfirst[lmax].as<int>(), sj.blast.as<int>(), sj.x.as<float>(),         \
      sj.y.as<float>(), sj.z.as<float>(), sj.nx.as<float>(), sj.ny.as<float>(), sj.nz.as<float>(), Q_,            \
      neq == FMMX_GNJ, cfg.convention, lmax, xmin, ymin, zmin, rb(lmax), corr, mexp[lmax].as<T_>(), lrb, STRIDE_, \
      OFF_, qs2.as<float>())
    // Laplace charges in the EXACT convention: the streaming form
#define FMMX_P2M_H(T_, YK_, H_, Q_, STRIDE_, OFF_)                                                 \
  do {                                                                                            \
    if constexpr (YK_ == 0) {                                                                     \
      if (neq != FMMX_GNJ && cfg.convention == FMMX_CONV_EXACT && std::is_same_v<T_, float>)      \
        k_p2m_exact<P, H_><<<H_ ? (nb + 1) / 2 : nb, 64, 0, stream>>>(                            \
            nb, sj.bkey[lmax].as<uint32_t>(), sj.bfirst[lmax].as<int>(), sj.blast.as<int>(),      \
            sj.x.as<float>(), sj.y.as<float>(), sj.z.as<float>(), Q_, lmax, xmin, ymin, zmin,     \
            rb(lmax), (float*)mexp[lmax].as<T_>(), STRIDE_, OFF_);                                \
      else if (neq != FMMX_GNJ && cfg.convention == FMMX_CONV_EXACT)                              \
        FMMX_P2M_HC(T_, 0, H_, FMMX_CONV_EXACT, 0, Q_, STRIDE_, OFF_);                            \
      else                                                                                        \
        FMMX_P2M_HC(T_, 0, H_, -1, -1, Q_, STRIDE_, OFF_);                                        \
    } else {                                                                                      \
      FMMX_P2M_HC(T_, YK_, H_, -1, -1, Q_, STRIDE_, OFF_);                                        \
    }                                                                                             \
  } while (0)
#define FMMX_P2M(T_, YK_, Q_, STRIDE_, OFF_)                 \
  do {                                                       \
    if (half) FMMX_P2M_H(T_, YK_, 1, Q_, STRIDE_, OFF_);     \
    else FMMX_P2M_H(T_, YK_, 0, Q_, STRIDE_, OFF_);          \
  } while (0)
    if (hh) {
      // the multipoles of the real and of the imaginary charges, side by side
      if constexpr (P % 2 == 0 && P >= 4) {
        if (fp64) {
          FMMX_P2M(double, 2, qs.as<float>(), 2 * VS, 0);
        } else {
          FMMX_P2M(float, 2, qs.as<float>(), 2 * VS, 0);
        }
      } else {
        return fail(FMMX_EUNSUPPORTED, "Helmholtz needs p in {4, 6, 8, 10, 12}");
      }
    } else if (fp64) {
      if (yk) FMMX_P2M(double, 1, qs.as<float>(), VS, 0);
      else FMMX_P2M(double, 0, qs.as<float>(), VS, 0);
    } else {
      if (yk) FMMX_P2M(float, 1, qs.as<float>(), VS, 0);
      else FMMX_P2M(float, 0, qs.as<float>(), VS, 0);
    }
#undef FMMX_P2M
#undef FMMX_P2M_H
#undef FMMX_P2M_HC
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  });
}

}  // namespace fmmx
