// l2p.hip -- L2P (kernel/G_l2p.cxx, Gn_l2p.cxx) for CDNA4 (gfx950), wave64: one
// wave per leaf box (two leaves per wave when small); solid harmonics from a
// Cartesian recurrence; the outputs go out in the caller's order.
#include "phases.h"

namespace fmmx {

namespace {

// The far-field result of target i (sorted position) added to its near-field
// sums: stored back in place, or, with out.perm set, written straight to the
// caller's order (out.v[perm[i]], ...; the gradient outputs may be NULL),
// which saves the separate scatter pass over the outputs.
struct L2POut {
  const uint32_t* perm;
  double *v, *gx, *gy, *gz;
};
__device__ __forceinline__ void l2p_store(const L2POut& out, int i, int gn, int grad, double s1, double s2,
                                          double phi, double gx, double gy, double gz,
                                          const float* __restrict__ nx, const float* __restrict__ ny,
                                          const float* __restrict__ nz, double* __restrict__ vs,
                                          double* __restrict__ gxs, double* __restrict__ gys,
                                          double* __restrict__ gzs) {
  if (gn) {
    const double v = vs[i] - s2 * ((double)nx[i] * gx + (double)ny[i] * gy + (double)nz[i] * gz);
    if (!out.perm) vs[i] = v;
    else if (out.v) out.v[out.perm[i]] = v;
    return;
  }
  const double v = vs[i] + s1 * phi;
  if (!out.perm) {
    vs[i] = v;
    if (grad) {
      gxs[i] += s2 * gx;
      gys[i] += s2 * gy;
      gzs[i] += s2 * gz;
    }
    return;
  }
  const uint32_t j = out.perm[i];
  if (out.v) out.v[j] = v;
  if (grad) {
    if (out.gx) out.gx[j] = gxs[i] + s2 * gx;
    if (out.gy) out.gy[j] = gys[i] + s2 * gy;
    if (out.gz) out.gz[j] = gzs[i] + s2 * gz;
  }
}

// ---------------------------------------------------------------------
// L2P: one wave per target leaf box; adds to the P2P results (sorted order)
//   YK 1: Yukawa locals, phi = sum_n h_n(r) sum_m L~ S_n^m(u) with
//       h_n = i~_n(lambda r)/i~_n(lambda rb); grad adds
//       lrb^2 i~_{n+1}(lambda r)/i~_n(lambda rb) (sum_m L~ S_n^m) u
//   YK 2: one part (Re or Im of the field) of Helmholtz locals,
//       phi = c4/rb sum_n j^_n(k r) sum_m L S_n^m(u), potential only
//   Box b's local starts at L + b * lstride + loff.
template <int P, typename T, int YK = 0, int HALF = 0, int CONV = -1>
__global__ __launch_bounds__(64) void k_l2p(int nb, const uint32_t* __restrict__ bkey, const int* __restrict__ bfirst,
                                            const int* __restrict__ blast, const float* __restrict__ x,
                                            const float* __restrict__ y, const float* __restrict__ z,
                                            const float* __restrict__ nx, const float* __restrict__ ny,
                                            const float* __restrict__ nz, const T* __restrict__ L, int gn, int grad,
                                            int conv, int lev, double xmin, double ymin, double zmin, double rb,
                                            const double* __restrict__ corr, double c4, double* __restrict__ vs,
                                            double* __restrict__ gxs, double* __restrict__ gys,
                                            double* __restrict__ gzs, double lrb, int lstride, int loff,
                                            L2POut out) {
  // HALF: two leaves per wave (32 lanes each), for leaves of at most about
  // 32 targets where a whole wave per leaf would idle half its lanes
  constexpr int NR = P * (P + 1) / 2, P2 = P * P, NL = HALF ? 2 : 1, STEP = HALF ? 32 : 64;
  __shared__ T Lrs[NL][NR], Lis[NL][NR];
  const int h = HALF ? (int)(threadIdx.x >> 5) : 0, lane = HALF ? (int)(threadIdx.x & 31) : (int)threadIdx.x;
  const int b = HALF ? 2 * (int)blockIdx.x + h : (int)blockIdx.x;
  const bool valid = b < nb;
  T* Lr = Lrs[h];
  T* Li = Lis[h];
  // weights: 1 for m = 0, 2 for m > 0 (kernel/G_l2p.cxx:246-260); table ratio in REF
  for (int s = lane; valid && s < NR; s += STEP) {
    int n = 0;
    while (sl(n + 1, 0) <= s) n++;
    const int m = s - sl(n, 0);
    const double w = (m == 0 ? 1.0 : 2.0) * (YK ? 1.0 : corr[s]);
    Lr[s] = T(w * (double)L[(size_t)b * lstride + loff + s]);
    Li[s] = m == 0 ? T(0) : T(w * (double)L[(size_t)b * lstride + loff + NR + n * (n - 1) / 2 + m - 1]);
  }
  __syncthreads();
  if constexpr (YK == 0) {
    // The gradient of sum L_n^m S_n^m is a sum over S_{n-1}^{m'} with
    // coefficients linear in L (the derivative rules of the harmonics above),
    // so per leaf the table C[s] = (L, X/2, Y/2, Z) is built once and each
    // target streams its harmonics column by column against it, keeping only
    // the recurrence state live:
    //   gx = Re sum S X/2, gy = Im sum S Y/2, gz = Re sum S Z,
    //   X = gp(n,m-1) L_n^{m-1} - gm(n,m+1) L_n^{m+1} + [m=1] gp(n,0) conj(L_n^0),
    //   Y = gp(n,m-1) L_n^{m-1} + gm(n,m+1) L_n^{m+1} + [m=1] gp(n,0) conj(L_n^0),
    //   Z = gz(n,m) L_n^m, with n one above the degree of S.
    __shared__ __align__(16) T Cs[NL][NR][8];
    for (int s = lane; valid && s < NR; s += STEP) {
      int n = 0;
      while (sl(n + 1, 0) <= s) n++;
      const int m = s - sl(n, 0);
      T* c = Cs[h][s];
      c[0] = Lr[s];
      c[1] = Li[s];
      T xr = 0, xi = 0, yr = 0, yi = 0, zr = 0, zi = 0;
      if (n <= P - 2) {
        const int nu = n + 1;
        if (m >= 1) {
          const T g = T(c_hc.gp[nu][m - 1]), ar = g * Lr[sl(nu, m - 1)], ai = g * Li[sl(nu, m - 1)];
          xr += ar;
          xi += ai;
          yr += ar;
          yi += ai;
        }
        {
          const T g = T(c_hc.gm[nu][m + 1]), ar = g * Lr[sl(nu, m + 1)], ai = g * Li[sl(nu, m + 1)];
          xr -= ar;
          xi -= ai;
          yr += ar;
          yi += ai;
        }
        if (m == 1) {
          const T g = T(c_hc.gp[nu][0]), ar = g * Lr[sl(nu, 0)], ai = -g * Li[sl(nu, 0)];
          xr += ar;
          xi += ai;
          yr += ar;
          yi += ai;
        }
        const T g = T(c_hc.gz[nu][m]);
        zr = g * Lr[sl(nu, m)];
        zi = g * Li[sl(nu, m)];
      }
      c[2] = T(0.5) * xr;
      c[3] = T(0.5) * xi;
      c[4] = T(0.5) * yi;
      c[5] = T(0.5) * yr;
      c[6] = zr;
      c[7] = zi;
    }
    __syncthreads();
    const double rbinv = 1.0 / rb;
    // a compile-time convention keeps the REF angle code (double acos,
    // atan, sincos) out of the EXACT kernel's register budget
    const int cv = CONV >= 0 ? CONV : conv;
    // target i of the leaf whose table is Cs[hs], centre (cx, cy, cz)
    auto target = [&](int i, int hs, double cx, double cy, double cz) {
      double ux, uy, uz;
      eff_point(cv, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
      const T tx = T(ux), ty = T(uy), tz = T(uz), r2 = tx * tx + ty * ty + tz * tz;
      T phi = T(0), gx = T(0), gy = T(0), gz = T(0);
      // the table holds zero gradient entries at degree p-1
      auto term = [&](T sr, T si, int s) {
        const T* c = Cs[hs][s];
        phi += sr * c[0] - si * c[1];
        gx += sr * c[2] - si * c[3];
        gy += sr * c[4] + si * c[5];
        gz += sr * c[6] - si * c[7];
      };
      // harmonics column by column (runtime loops: only the recurrence state
      // is live, and the table reads cannot be hoisted out of the target loop)
      T dr = T(1), di = T(0);  // S_m^m
#pragma unroll 1
      for (int m = 0; m < P; m++) {
        if (m > 0) {
          const T a = -HC<T>::a(m), nr = a * (tx * dr - ty * di), ni = a * (tx * di + ty * dr);
          dr = nr;
          di = ni;
        }
        term(dr, di, sl(m, m));
        if (m + 1 < P) {
          const T bz = HC<T>::b(m) * tz;
          T pr = dr, pi = di, sr = bz * dr, si = bz * di;  // S_{n-1}^m, S_n^m
          term(sr, si, sl(m + 1, m));
#pragma unroll 1
          for (int n = m + 2; n < P; n++) {
            const T cz = HC<T>::c(n - 1, m) * tz, d = HC<T>::d(n - 1, m) * r2;
            const T nr = cz * sr - d * pr, ni = cz * si - d * pi;
            pr = sr;
            pi = si;
            sr = nr;
            si = ni;
            term(sr, si, sl(n, m));
          }
        }
      }
      l2p_store(out, i, gn, grad, c4 * rbinv, c4 * rbinv * rbinv, (double)phi, (double)gx, (double)gy, (double)gz, nx, ny,
                nz, vs, gxs, gys, gzs);
    };
    if constexpr (HALF != 0) {
      // the targets of the wave's two leaves, one list over all 64 lanes: a
      // leaf of 33-40 targets beside a smaller one still takes one pass
      const int bA = 2 * (int)blockIdx.x, bB = bA + 1;  // bA < nb: the grid is (nb + 1) / 2
      const int a0 = bfirst[bA], nA = max(0, blast[bA] - a0 + 1);
      const bool vB = bB < nb;
      const int b0 = vB ? bfirst[bB] : 0, nB = vB ? max(0, blast[bB] - b0 + 1) : 0;
      double axc, ayc, azc, bxc = 0, byc = 0, bzc = 0;
      box_center(bkey[bA], lev, xmin, ymin, zmin, rb, axc, ayc, azc);
      if (vB) box_center(bkey[bB], lev, xmin, ymin, zmin, rb, bxc, byc, bzc);
      for (int t = (int)threadIdx.x; t < nA + nB; t += 64) {
        const bool hb = t >= nA;
        target(hb ? b0 + (t - nA) : a0 + t, hb ? 1 : 0, hb ? bxc : axc, hb ? byc : ayc, hb ? bzc : azc);
      }
    } else {
      if (!valid) return;
      double cx, cy, cz;
      box_center(bkey[b], lev, xmin, ymin, zmin, rb, cx, cy, cz);
      const int i0 = bfirst[b], i1 = blast[b];
      for (int i = i0 + lane; i <= i1; i += STEP) target(i, h, cx, cy, cz);
    }
    return;
  }
  if (!valid) return;
  double cx, cy, cz;
  box_center(bkey[b], lev, xmin, ymin, zmin, rb, cx, cy, cz);
  const double rbinv = 1.0 / rb;
  const int i0 = bfirst[b], i1 = blast[b];
  for (int i = i0 + lane; i <= i1; i += STEP) {
    double ux, uy, uz;
    eff_point(conv, (double)x[i] - cx, (double)y[i] - cy, (double)z[i] - cz, rbinv, ux, uy, uz);
    T Sr[NR], Si[NR];
    solid_harmonics<P, T>(T(ux), T(uy), T(uz), Sr, Si);
    T phi = T(0), gx = T(0), gy = T(0), gz = T(0);
    if constexpr (YK == 2) {
      double jn[P];
      jhat_dev<P - 1>(lrb * sqrt(ux * ux + uy * uy + uz * uz), jn);
#pragma unroll
      for (int n = 0; n < P; n++) {
        T pn = T(0);
#pragma unroll
        for (int m = 0; m <= n; m++) pn += Sr[sl(n, m)] * Lr[sl(n, m)] - Si[sl(n, m)] * Li[sl(n, m)];
        phi += T(jn[n]) * pn;
      }
    } else if constexpr (YK) {
      double hn[P + 1], h0[P];
      ibar_dev<P - 1>(lrb, h0);
      ibar_dev<P>(lrb * sqrt(ux * ux + uy * uy + uz * uz), hn);
#pragma unroll
      for (int n = 0; n < P; n++) {
        T pn = T(0), gxn = T(0), gyn = T(0), gzn = T(0);
#pragma unroll
        for (int m = 0; m <= n; m++) {
          const int s = sl(n, m);
          const T lr = Lr[s], li = Li[s];
          pn += Sr[s] * lr - Si[s] * li;
          if (n >= 1) {
            T pr, pi, mr, mi, zr, zi;
            harm_grad<P, T>(Sr, Si, n, m, pr, pi, mr, mi, zr, zi);
            const T apr = pr * lr - pi * li, api = pr * li + pi * lr;
            const T amr = mr * lr - mi * li, ami = mr * li + mi * lr;
            gxn += T(0.5) * (apr + amr);
            gyn += T(0.5) * (api - ami);
            gzn += zr * lr - zi * li;
          }
        }
        const T h = T(hn[n] / h0[n]), e = T(lrb * lrb * hn[n + 1] / h0[n]) * pn;
        phi += h * pn;
        gx += h * gxn + e * T(ux);
        gy += h * gyn + e * T(uy);
        gz += h * gzn + e * T(uz);
      }
    } else {
#pragma unroll
      for (int n = 0; n < P; n++)
#pragma unroll
        for (int m = 0; m <= n; m++) {
          const int s = sl(n, m);
          const T lr = Lr[s], li = Li[s];
          phi += Sr[s] * lr - Si[s] * li;
          if (n >= 1) {
            T pr, pi, mr, mi, zr, zi;
            harm_grad<P, T>(Sr, Si, n, m, pr, pi, mr, mi, zr, zi);
            // Re(Ap L), Im(Ap L), Re(Am L), Im(Am L)
            const T apr = pr * lr - pi * li, api = pr * li + pi * lr;
            const T amr = mr * lr - mi * li, ami = mr * li + mi * lr;
            gx += T(0.5) * (apr + amr);
            gy += T(0.5) * (api - ami);
            gz += zr * lr - zi * li;
          }
        }
    }
    l2p_store(out, i, gn, grad, c4 * rbinv, c4 * rbinv * rbinv, (double)phi, (double)gx, (double)gy, (double)gz, nx, ny,
              nz, vs, gxs, gys, gzs);
  }
}

}  // namespace

int Engine::run_l2p(int neq, double* const* dst) {
  const int nb = si.nb[lmax];
  if (nb == 0) return FMMX_OK;
  // with dst (v, gx, gy, gz in the caller's order) the results go there
  L2POut lout{};
  if (dst && !hh) lout = L2POut{si.perm.as<uint32_t>(), dst[0], dst[1], dst[2], dst[3]};
  const double* corr = corr_d.as<double>();
  if (p > P_ALL) {
    return dispatch_hi(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value;
      const double lrb = lam * rb(lmax), cl = yk ? rb(lmax) : c4();
      const int grad = neq == FMMX_G || neq == FMMX_YUKAWA;
#define FMMX_L2P_HI(YK_, C_)                                                                                    \
  k_l2p<P, double, YK_, 0, C_><<<nb, 64, 0, stream>>>(                                                          \
      nb, si.bkey[lmax].as<uint32_t>(), si.bfirst[lmax].as<int>(), si.blast.as<int>(), si.x.as<float>(),      \
      si.y.as<float>(), si.z.as<float>(), si.nx.as<float>(), si.ny.as<float>(), si.nz.as<float>(),             \
      lexp[lmax].as<double>(), neq == FMMX_GNI, grad, cfg.convention, lmax, xmin, ymin, zmin, rb(lmax), corr, \
      cl, vs.as<double>(), gxs.as<double>(), gys.as<double>(), gzs.as<double>(), lrb, P * P, 0, lout)
      if (yk) FMMX_L2P_HI(1, -1);
      else FMMX_L2P_HI(0, FMMX_CONV_EXACT);
#undef FMMX_L2P_HI
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  return dispatch_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    // Yukawa locals carry the kernel's constant: phi = sum L~ h_n S_n(u)
    const double lrb = (hh ? hk : lam) * rb(lmax), cl = yk ? rb(lmax) : c4();
    const int grad = neq == FMMX_G || neq == FMMX_YUKAWA;
    // two leaves per wave when leaves hold at most about 32 targets
    const bool half = (double)si.n / nb <= 32.0;
#define FMMX_L2P_HC(T_, YK_, H_, C_, V_, STRIDE_, OFF_)                                                           \
  k_l2p<P, T_, YK_, H_, C_><<<H_ ? (nb + 1) / 2 : nb, 64, 0, stream>>>(                                          \
      nb, si.bkey[lmax].as<uint32_t>(), si.bfirst[lmax].as<int>(), si.blast.as<int>(), si.x.as<float>(),        \
      si.y.as<float>(), si.z.as<float>(), si.nx.as<float>(), si.ny.as<float>(), si.nz.as<float>(),               \
      lexp[lmax].as<T_>(), neq == FMMX_GNI, grad, cfg.convention, lmax, xmin, ymin, zmin, rb(lmax), corr, cl, V_, \
      gxs.as<double>(), gys.as<double>(), gzs.as<double>(), lrb, STRIDE_, OFF_, lout)
    // Laplace: the convention as a template argument
#define FMMX_L2P_H(T_, YK_, H_, V_, STRIDE_, OFF_)                                          \
  do {                                                                                     \
    if constexpr (YK_ != 0) FMMX_L2P_HC(T_, YK_, H_, -1, V_, STRIDE_, OFF_);               \
    else if (cfg.convention == FMMX_CONV_REF)                                              \
      FMMX_L2P_HC(T_, 0, H_, FMMX_CONV_REF, V_, STRIDE_, OFF_);                            \
    else FMMX_L2P_HC(T_, 0, H_, FMMX_CONV_EXACT, V_, STRIDE_, OFF_);                       \
  } while (0)
#define FMMX_L2P(T_, YK_, V_, STRIDE_, OFF_)               \
  do {                                                     \
    if (half) FMMX_L2P_H(T_, YK_, 1, V_, STRIDE_, OFF_);   \
    else FMMX_L2P_H(T_, YK_, 0, V_, STRIDE_, OFF_);        \
  } while (0)
    if (hh) {
      // Re of the potential into vs, Im into gxs
      if constexpr (P % 2 == 0 && P >= 4) {
        if (fp64) {
          FMMX_L2P(double, 2, vs.as<double>(), 2 * P2, 0);
          FMMX_L2P(double, 2, gxs.as<double>(), 2 * P2, P2);
        } else {
          FMMX_L2P(float, 2, vs.as<double>(), 2 * P2, 0);
          FMMX_L2P(float, 2, gxs.as<double>(), 2 * P2, P2);
        }
      } else {
        return fail(FMMX_EUNSUPPORTED, "Helmholtz needs p in {4, 6, 8, 10, 12}");
      }
    } else if (fp64) {
      if (yk) FMMX_L2P(double, 1, vs.as<double>(), P2, 0);
      else FMMX_L2P(double, 0, vs.as<double>(), P2, 0);
    } else {
      if (yk) FMMX_L2P(float, 1, vs.as<double>(), P2, 0);
      else FMMX_L2P(float, 0, vs.as<double>(), P2, 0);
    }
#undef FMMX_L2P
#undef FMMX_L2P_H
#undef FMMX_L2P_HC
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  });
}

}  // namespace fmmx
