// The host side of the orbit M2L (split_host.cpp) built with AddressSanitizer and
// UndefinedBehaviorSanitizer: the orbits of every parity class against the
// interaction list, and the operator fragments of the three kernels multiplied
// as the kernels do against the dense operators, for every order built.
#include <algorithm>
#include <array>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <set>
#include <type_traits>
#include <vector>

#include "../../old_fmm_bem_amd/csrc/fmmx_internal.h"
#include "../../old_fmm_bem_amd/csrc/helmholtz.h"
#include "../../old_fmm_bem_amd/csrc/m2l.h"

using namespace fmmx;

static int bad = 0;
static void check(bool ok, const char* what, int p) {
  if (!ok) std::printf("%s at p = %d\n", what, p), bad++;
}

static double half(uint32_t h) {
  const int e = (h >> 10) & 31;
  const double m = h & 1023, v = e ? std::ldexp(1 + m / 1024, e - 15) : std::ldexp(m, -24);
  return h & 0x8000 ? -v : v;
}
static double word(const uint4& f, int t) {
  const uint32_t w[4] = {f.x, f.y, f.z, f.w};
  return half((w[t / 2] >> (16 * (t & 1))) & 0xffff);
}

static std::mt19937 gen(1);
static std::vector<double> random(size_t n) {
  std::uniform_real_distribution<double> u(-1, 1);
  std::vector<double> x(n);
  for (double& v : x) v = u(gen);
  return x;
}

// largest difference of y from A x (row-major A), over the largest row sum of |A|
static double off(const std::vector<double>& y, const double* A, const std::vector<double>& x) {
  const int n = (int)x.size();
  double d = 0, s = 0;
  for (int i = 0; i < n; i++) {
    double v = 0, m = 0;
    for (int k = 0; k < n; k++) v += A[(size_t)i * n + k] * x[k], m += std::fabs(A[(size_t)i * n + k]);
    d = std::max(d, std::fabs(v - y[i]));
    s = std::max(s, m);
  }
  return d / s;
}

static void orbits() {
  std::set<int> used;
  for (int cls = 0; cls < 8; cls++) {
    std::set<std::array<int, 3>> seen;
    for (int o = 0; o < NORB; o++) {
      int d[3];
      orbit_offset(o, cls, d);
      const int D = orb_mask(o), op = orbit_op_index(d);
      check(op >= 0 && op < NORBOP, "operator of an orbit", o);
      check(orb_start(D) <= o && o < orb_start(D + 1), "mask of an orbit", o);
      used.insert(op);
      for (int r = 0; r < 8; r++) {
        if (r & ~D) continue;
        std::array<int, 3> e;
        for (int a = 0; a < 3; a++) e[a] = (r >> a) & 1 ? -d[a] : d[a];
        check(seen.insert(e).second, "offset in two orbits", o);
      }
    }
    size_t n = 0;
    for (int dx = -3; dx <= 3; dx++)
      for (int dy = -3; dy <= 3; dy++)
        for (int dz = -3; dz <= 3; dz++) {
          const int d[3] = {dx, dy, dz};
          bool in = std::max({std::abs(dx), std::abs(dy), std::abs(dz)}) > 1;
          for (int a = 0; a < 3; a++) in = in && d[a] >= ((cls >> a) & 1) - 3 && d[a] <= ((cls >> a) & 1) + 2;
          n += in;
          check(!in || seen.count({dx, dy, dz}), "offset of the interaction list without an orbit", cls);
        }
    check(n == seen.size() && n == 189, "offsets of a class", cls);
  }
  check((int)used.size() == NORBOP, "operators used", 0);
}

struct Laplace {
  std::vector<double> kmaj;
  explicit Laplace(int p) : kmaj((size_t)NOFF * p * p * p * p) {
    Tables T;
    build_tables(T, p, FMMX_CONV_EXACT);
    const int P2 = p * p;
    std::vector<double> A((size_t)P2 * P2);
    for (int o = 0; o < NOFF; o++) {
      int d[3];
      offset_vector(o, d);
      op_m2l(T, d[0], d[1], d[2], 1.0, A.data());
      for (int r = 0; r < P2; r++)
        for (int k = 0; k < P2; k++) kmaj[((size_t)o * P2 + k) * P2 + r] = A[(size_t)r * P2 + k];
    }
  }
  // operator i of the orbits, row-major
  std::vector<double> op(int i, int p) const {
    int d[3];
    orbit_op_vector(i, d);
    const int P2 = p * p, o = offset_index(d[0], d[1], d[2]);
    std::vector<double> A((size_t)P2 * P2);
    for (int r = 0; r < P2; r++)
      for (int k = 0; k < P2; k++) A[(size_t)r * P2 + k] = kmaj[((size_t)o * P2 + k) * P2 + r];
    return A;
  }
};

// hi + lo of FP16 hold 22 bits; 2^-20 of the largest row sum allows for the
// smallest steps of small elements
constexpr double TOL16 = 1.0 / (1 << 20);

template <int P>
void mixed(const Laplace& L) {
  using OC = OConst<P>;
  constexpr OLayout<P> O{};
  const int e = split_scale_exp(L.kmaj.data(), L.kmaj.size());
  std::vector<uint4> f;
  orbit_fragments(L.kmaj.data(), P, e, f);
  check(f.size() == (size_t)NORBOP * OC::FRO, "orbit fragments", P);
  check(orbit_box_floats(P) == (size_t)OC::BS, "orbit box", P);
  for (int i = 0; i < NORBOP; i += 41) {
    const std::vector<double> x = random(P * P);
    std::vector<double> y(P * P, 0.0);
    const uint4* A = &f[(size_t)i * OC::FRO];
    for (int s = 0; s < OC::NSTEP; s++)
      for (int c = 0; c < 8; c++)
        for (int l = 0; l < 64; l++) {
          if (O.slot[c][l & 15] < 0) continue;
          double v = 0;
          for (int t = 0; t < 8; t++) {
            const bool q = s == OC::NO;
            const int k = q ? O.qc[t & 3] : t, m = 4 * s + (l >> 4);
            if (m >= O.size[k]) continue;
            const double a = q ? word(A[OC::NO * OC::FRS + c * 64 + l], t)
                               : word(A[s * OC::FRS + 2 * c * 64 + l], t) + word(A[s * OC::FRS + (2 * c + 1) * 64 + l], t);
            v += a * x[O.slot[k][m]];
          }
          y[O.slot[c][l & 15]] += std::ldexp(v, -e);
        }
    check(off(y, L.op(i, P).data(), x) < TOL16, "orbit product", P);
  }
}

template <int P>
void fp64(const Laplace& L) {
  using F = FConst<P>;
  constexpr GLayout<P> G{};
  std::vector<double> f;
  orbit_f64_fragments(L.kmaj.data(), P, f);
  check(f.size() == (size_t)NORBOP * F::FRO * 2, "FP64 orbit fragments", P);
  check(orbit_f64_box(P) == (size_t)F::BS && orbit_f64_rows(P) == (size_t)F::ROWS, "FP64 orbit sizes", P);
  for (int i = 0; i < NORBOP; i += 41) {
    const std::vector<double> x = random(P * P);
    std::vector<double> y(P * P, 0.0);
    for (int ks = 0; ks < F::NKS; ks++)
      for (int tl = 0; tl < F::NT; tl++)
        for (int l = 0; l < 64; l++) {
          const int r = G.trow[tl] + 4 * (l & 3) + ((l & 15) >> 2), m = G.member(F::step(ks), F::place(ks), l >> 4);
          if (r >= G.O.size[G.tcls[tl]] || m < 0) continue;
          const double a = f[(size_t)i * F::FRO * 2 + (((size_t)ks / 2 * F::NT + tl) * 64 + l) * 2 + (ks & 1)];
          y[G.O.slot[G.tcls[tl]][r]] += a * x[G.O.slot[G.cls(F::step(ks), F::place(ks))][m]];
        }
    check(off(y, L.op(i, P).data(), x) < 1e-14, "FP64 orbit product", P);
  }
}

template <int P>
void helmholtz() {
  using GC = GConst<P>;
  constexpr GLayout<P> G{};
  constexpr int P2 = P * P;
  check(orbit_gen_box_floats(P) == (size_t)GC::BS && orbit_gen_frags(P) == (size_t)GC::FRO &&
            orbit_gen_rows(P) == (size_t)GC::ROWS, "Helmholtz orbit sizes", P);
  std::vector<double> H((size_t)4 * P2 * P2), C((size_t)P2 * P2), S(C.size());
  std::vector<uint4> f(orbit_gen_frags(P));
  for (double kappa : {0.01, 1.3, 4.9}) {
    hh_op_m2l(P, kappa, 2, 1, -3, H.data());
    for (int r = 0; r < P2; r++)
      for (int k = 0; k < P2; k++) {
        C[(size_t)r * P2 + k] = H[(size_t)r * 2 * P2 + k];
        S[(size_t)r * P2 + k] = H[(size_t)(P2 + r) * 2 * P2 + k];
      }
    const int e = std::min(split_scale_exp(C.data(), C.size()), split_scale_exp(S.data(), S.size()));
    orbit_gen_fragments(C.data(), S.data(), P2, P, e, f.data());
    for (int q = 0; q < 2; q++) {
      const std::vector<double> x = random(P2);
      std::vector<double> y(P2, 0.0);
      for (int s = 0; s < GC::NSTEP; s++)
        for (int tl = 0; tl < GC::NT; tl++)
          for (int l = 0; l < 64; l++) {
            const int r = G.trow[tl] + (l & 15);
            if (r >= G.O.size[G.tcls[tl]]) continue;
            const uint4* A = &f[(((size_t)s * GC::NT + tl) * 2 + q) * 2 * 64 + l];
            double v = 0;
            for (int t = 0; t < 8; t++) {
              const int m = G.member(s, t, l >> 4);
              if (m >= 0) v += (word(A[0], t) + word(A[64], t)) * x[G.O.slot[G.cls(s, t)][m]];
            }
            y[G.O.slot[G.tcls[tl]][r]] += std::ldexp(v, -e);
          }
      // both blocks share the scale of the larger
      double big = 0, own = 0;
      for (int r = 0; r < P2; r++) {
        double a = 0, b = 0;
        for (int k = 0; k < P2; k++) a += std::fabs(C[(size_t)r * P2 + k]), b += std::fabs(S[(size_t)r * P2 + k]);
        big = std::max({big, a, b});
        own = std::max(own, q ? b : a);
      }
      check(off(y, (q ? S : C).data(), x) * own / big < TOL16, "Helmholtz orbit product", P);
    }
  }
}

template <int P>
void laplace() {
  const Laplace L(P);
  if constexpr (P <= 10) mixed<P>(L);
  fp64<P>(L);
}

int main() {
  orbits();
  laplace<6>();
  laplace<7>();
  laplace<8>();
  laplace<9>();
  laplace<10>();
  laplace<11>();
  laplace<12>();
  helmholtz<4>();
  helmholtz<6>();
  helmholtz<8>();
  helmholtz<10>();
  helmholtz<12>();
  std::printf("orbit checks: %d failures\n", bad);
  return bad ? 1 : 0;
}
