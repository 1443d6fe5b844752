// split_host.cpp -- host side of the error-compensated FP16 M2L
// (m2l_split.hip): the operators' FP16 hi/lo split in the kernels' fragment
// orders and the power-of-two scale that keeps them in range.  Plain host
// C++ (no device code), so that it also builds under the sanitizers.
#include <algorithm>
#include <array>
#include <cmath>
#include <type_traits>
#include <vector>

#include "m2l.h"

namespace fmmx {

namespace {

// IEEE binary16 of x, rounded to nearest even (host)
uint16_t to_half(double x) {
  const uint16_t sgn = std::signbit(x) ? 0x8000 : 0;
  double a = std::fabs(x);
  if (a == 0.0) return sgn;
  if (!(a < 65520.0)) return sgn | 0x7c00;
  int e;
  (void)std::frexp(a, &e);  // a = m 2^e, m in [0.5, 1)
  const int ex = e - 1;      // a in [2^ex, 2^(ex+1))
  if (ex < -14) return sgn | (uint16_t)std::nearbyint(std::ldexp(a, 24));  // subnormal (1024: smallest normal)
  double q = std::nearbyint(std::ldexp(a, 10 - ex));
  int be = ex + 15;
  if (q >= 2048.0) {
    q = 1024.0;
    be++;
  }
  if (be >= 31) return sgn | 0x7c00;
  return sgn | (uint16_t)(be << 10) | (uint16_t)(q - 1024.0);
}

double from_half(uint16_t h) {
  const int be = (h >> 10) & 31, mant = h & 1023;
  const double v = be == 0 ? std::ldexp((double)mant, -24) : std::ldexp(1024.0 + mant, be - 25);
  return (h & 0x8000) ? -v : v;
}

}  // namespace

// two operator buffers of the 32x32x16 form fit one CU's LDS
bool split_wide_fits(int p) {
  if (p < 6 || p > 12) return false;
  const int P2 = p * p, MT = (P2 + 31) / 32, KS = (P2 + 1) / 2, SEG = KS + (KS & 1), KH = (3 * SEG + 7) / 8;
  return (size_t)2 * KH * MT * 64 * 16 <= 160 * 1024 - 64;
}

// two operator buffers of the 16x16x32 form fit one CU's LDS
bool split_db_fits(int p) {
  const int P2 = p * p, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, SEG = KS + (KS & 1), KH = (3 * SEG + 7) / 8;
  return (size_t)2 * KH * MT * 64 * 16 <= 160 * 1024 - 64;
}

int split_scale_exp(const double* ops, size_t n) {
  double mx = 0;
  for (size_t i = 0; i < n; i++) mx = std::max(mx, std::fabs(ops[i]));
  if (!(mx > 0)) return 0;
  int e;
  (void)std::frexp(mx, &e);
  return SPLIT_TOP - e;
}

void split_fragments(const double* kmaj, int count, int p, int sa_e, std::vector<uint4>& out) {
  const int P2 = p * p, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, SEG = KS + (KS & 1), KH = (3 * SEG + 7) / 8;
  const size_t FRH = (size_t)KH * MT * 64;
  out.assign((size_t)count * FRH, make_uint4(0u, 0u, 0u, 0u));
  for (int o = 0; o < count; o++) {
    const double* A = kmaj + (size_t)o * P2 * P2;  // element (i, k) at A[k * P2 + i]
    for (int ks = 0; ks < KH; ks++)
      for (int mt = 0; mt < MT; mt++)
        for (int l = 0; l < 64; l++) {
          const int i = 16 * mt + (l & 15), g = l >> 4;
          uint16_t h[8] = {};
          for (int t = 0; t < 8; t++) {
            const int s = 8 * ks + t, seg = s / SEG, u = s % SEG, k = g * KS + u;
            if (i >= P2 || seg >= 3 || u >= KS || k >= P2) continue;
            const double a = std::ldexp(A[(size_t)k * P2 + i], sa_e);
            const uint16_t hi = to_half(a);
            h[t] = seg == 1 ? to_half(a - from_half(hi)) : hi;
          }
          out[(size_t)o * FRH + ((size_t)ks * MT + mt) * 64 + l] =
              make_uint4(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16, h[4] | (uint32_t)h[5] << 16,
                         h[6] | (uint32_t)h[7] << 16);
        }
  }
}

void split_fragments_wide(const double* kmaj, int count, int p, int sa_e, std::vector<uint4>& out) {
  const int P2 = p * p, MT = (P2 + 31) / 32, KS = (P2 + 1) / 2, SEG = KS + (KS & 1), KH = (3 * SEG + 7) / 8;
  const size_t FRW = (size_t)KH * MT * 64;
  out.assign((size_t)count * FRW, make_uint4(0u, 0u, 0u, 0u));
  for (int o = 0; o < count; o++) {
    const double* A = kmaj + (size_t)o * P2 * P2;  // element (i, k) at A[k * P2 + i]
    for (int ks = 0; ks < KH; ks++)
      for (int mt = 0; mt < MT; mt++)
        for (int l = 0; l < 64; l++) {
          const int i = 32 * mt + (l & 31), g = l >> 5;
          uint16_t h[8] = {};
          for (int t = 0; t < 8; t++) {
            const int s = 8 * ks + t, seg = s / SEG, u = s % SEG, k = g * KS + u;
            if (i >= P2 || seg >= 3 || u >= KS || k >= P2) continue;
            const double a = std::ldexp(A[(size_t)k * P2 + i], sa_e);
            const uint16_t hi = to_half(a);
            h[t] = seg == 1 ? to_half(a - from_half(hi)) : hi;
          }
          out[(size_t)o * FRW + ((size_t)ks * MT + mt) * 64 + l] =
              make_uint4(h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16, h[4] | (uint32_t)h[5] << 16,
                         h[6] | (uint32_t)h[7] << 16);
        }
  }
}

// ---- reflection orbits ------------------------------------------------
bool m2l_orbit_supported(int p) { return p >= 6 && p <= 10; }

namespace {
template <class F>
auto with_orbit_p(int p, F&& f) {
  switch (p) {
    case 6: return f(OConst<6>{}, std::integral_constant<int, 6>{});
    case 7: return f(OConst<7>{}, std::integral_constant<int, 7>{});
    case 8: return f(OConst<8>{}, std::integral_constant<int, 8>{});
    case 9: return f(OConst<9>{}, std::integral_constant<int, 9>{});
    default: return f(OConst<10>{}, std::integral_constant<int, 10>{});
  }
}
}  // namespace

void orbit_offset(int o, int cls, int* d) {
  // axis a in D: component 1 or 2 (both signs), else 0 or +-3 (the sign a
  // target of this parity sees); bit a of the choice picks the larger, and the
  // choice 0 (every |component| at most 1) is the near field
  const int D = orb_mask(o), k = o - orb_start(D), half = k / 7, pick = k % 7 + 1;
  const int axes = half > 0 ? 7 : D;  // the halves: z doubled too, one sign each
  for (int a = 0; a < 3; a++) {
    const int big = (pick >> a) & 1;
    if ((axes >> a) & 1) d[a] = 1 + big;
    else d[a] = !big ? 0 : (cls >> a) & 1 ? 3 : -3;
  }
  if (half == 2) d[2] = -d[2];
}

namespace {
// the distinct base offsets over all classes, in order of first appearance
const std::vector<std::array<int, 3>>& orbit_ops() {
  static const std::vector<std::array<int, 3>> v = [] {
    std::vector<std::array<int, 3>> u;
    for (int cls = 0; cls < 8; cls++)
      for (int o = 0; o < NORB; o++) {
        std::array<int, 3> d;
        orbit_offset(o, cls, d.data());
        if (std::find(u.begin(), u.end(), d) == u.end()) u.push_back(d);
      }
    return u;
  }();
  return v;
}
}  // namespace

int orbit_op_index(const int* d) {
  const auto& u = orbit_ops();
  const auto it = std::find(u.begin(), u.end(), std::array<int, 3>{d[0], d[1], d[2]});
  return it == u.end() ? -1 : (int)(it - u.begin());
}

size_t orbit_box_floats(int p) {
  if (!m2l_orbit_supported(p)) return 0;
  return with_orbit_p(p, [](auto oc, auto) -> size_t { return decltype(oc)::BS; });
}

void orbit_fragments(const double* kmaj, int p, int sa_e, std::vector<uint4>& out) {
  with_orbit_p(p, [&](auto oc, auto pc) -> int {
    using OC = decltype(oc);
    constexpr int P2 = decltype(pc)::value * decltype(pc)::value;
    const auto& O = OC::O;
    out.assign((size_t)NORBOP * OC::FRO, make_uint4(0u, 0u, 0u, 0u));
    const auto& ops = orbit_ops();
    for (size_t oi = 0; oi < ops.size(); oi++) {
      const double* A = kmaj + (size_t)offset_index(ops[oi][0], ops[oi][1], ops[oi][2]) * P2 * P2;  // (i, k) at [k P2 + i]
      uint4* dst = &out[oi * OC::FRO];
      for (int s = 0; s < OC::NSTEP; s++)
        for (int c = 0; c < 8; c++)
          for (int l = 0; l < 64; l++) {
            const int i = O.slot[c][l & 15], g = l >> 4;
            uint16_t h[2][8] = {};
            for (int t = 0; t < 8; t++) {
              const bool q = s == OC::NO;  // the quad step: hi words, lo words
              const int kc = q ? O.qc[t & 3] : t, mem = 4 * s + g;
              const int k = mem < O.size[kc] ? O.slot[kc][mem] : -1;
              if (i < 0 || k < 0) continue;
              const double a = std::ldexp(A[(size_t)k * P2 + i], sa_e);
              const uint16_t hi = to_half(a), lo = to_half(a - from_half(hi));
              h[0][t] = q && t >= 4 ? lo : hi;
              h[1][t] = lo;
            }
            auto frag = [&](int e) {
              return make_uint4(h[e][0] | (uint32_t)h[e][1] << 16, h[e][2] | (uint32_t)h[e][3] << 16,
                                h[e][4] | (uint32_t)h[e][5] << 16, h[e][6] | (uint32_t)h[e][7] << 16);
            };
            if (s < OC::NO) {
              for (int e = 0; e < 2; e++) dst[s * OC::FRS + (c * 2 + e) * 64 + l] = frag(e);
            } else {
              dst[OC::NO * OC::FRS + c * 64 + l] = frag(0);
            }
          }
    }
    return 0;
  });
}

void orbit_op_vector(int i, int* d) {
  for (int a = 0; a < 3; a++) d[a] = orbit_ops()[i][a];
}

namespace {
template <int P>
size_t gen_size(int what) {
  using G = GConst<P>;
  return what == 0 ? G::BS : what == 1 ? G::FRO : G::ROWS;
}
size_t gen_size(int p, int what) {
  switch (p) {
    case 4: return gen_size<4>(what);
    case 6: return gen_size<6>(what);
    case 8: return gen_size<8>(what);
    case 10: return gen_size<10>(what);
    case 12: return gen_size<12>(what);
  }
  return 0;
}
template <int P>
void gen_fragments(const double* C, const double* S, int ld, int sa_e, uint4* out) {
  constexpr GLayout<P> L{};
  for (int s = 0; s < L.no + L.xtra; s++)
    for (int tl = 0; tl < L.nt; tl++)
      for (int q = 0; q < 2; q++)
        for (int l = 0; l < 64; l++) {
          const double* A = q ? S : C;
          const int r = L.trow[tl] + (l & 15), i = r < L.O.size[L.tcls[tl]] ? L.O.slot[L.tcls[tl]][r] : -1;
          uint16_t h[2][8] = {};
          for (int t = 0; t < 8; t++) {
            const int m = L.member(s, t, l >> 4);
            if (i < 0 || m < 0) continue;
            const double a = std::ldexp(A[(size_t)i * ld + L.O.slot[L.cls(s, t)][m]], sa_e);
            h[0][t] = to_half(a);
            h[1][t] = to_half(a - from_half(h[0][t]));
          }
          for (int e = 0; e < 2; e++)
            out[((((size_t)s * L.nt + tl) * 2 + q) * 2 + e) * 64 + l] =
                make_uint4(h[e][0] | (uint32_t)h[e][1] << 16, h[e][2] | (uint32_t)h[e][3] << 16,
                           h[e][4] | (uint32_t)h[e][5] << 16, h[e][6] | (uint32_t)h[e][7] << 16);
        }
}
}  // namespace

size_t orbit_gen_box_floats(int p) { return gen_size(p, 0); }
size_t orbit_gen_frags(int p) { return gen_size(p, 1); }
size_t orbit_gen_rows(int p) { return gen_size(p, 2); }

void orbit_gen_fragments(const double* C, const double* S, int ld, int p, int sa_e, uint4* out) {
  switch (p) {
    case 4: return gen_fragments<4>(C, S, ld, sa_e, out);
    case 6: return gen_fragments<6>(C, S, ld, sa_e, out);
    case 8: return gen_fragments<8>(C, S, ld, sa_e, out);
    case 10: return gen_fragments<10>(C, S, ld, sa_e, out);
    case 12: return gen_fragments<12>(C, S, ld, sa_e, out);
  }
}

namespace {
template <typename G>
auto with_f64(int p, G&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(6) FMMX_CASE(7) FMMX_CASE(8) FMMX_CASE(9) FMMX_CASE(10) FMMX_CASE(11)
#undef FMMX_CASE
  }
  return f(std::integral_constant<int, 12>{});
}
}  // namespace

size_t orbit_f64_box(int p) {
  return with_f64(p, [](auto pc) -> size_t { return FConst<decltype(pc)::value>::BS; });
}
size_t orbit_f64_rows(int p) {
  return with_f64(p, [](auto pc) -> size_t { return FConst<decltype(pc)::value>::ROWS; });
}
void orbit_f64_fragments(const double* kmaj, int p, std::vector<double>& out) {
  with_f64(p, [&](auto pc) {
    constexpr int P = decltype(pc)::value, P2 = P * P;
    using F = FConst<P>;
    constexpr GLayout<P> L{};
    const auto& ops = orbit_ops();
    out.assign((size_t)NORBOP * F::FRO * 2, 0.0);
    for (size_t oi = 0; oi < ops.size(); oi++) {
      const double* A = kmaj + (size_t)offset_index(ops[oi][0], ops[oi][1], ops[oi][2]) * P2 * P2;  // (i, k) at [k P2 + i]
      double* dst = &out[oi * F::FRO * 2];
      for (int ks = 0; ks < F::NKS; ks++)
        for (int tl = 0; tl < F::NT; tl++)
          for (int l = 0; l < 64; l++) {
            // row rho of v_mfma_f64_16x16x4 comes out in lane group rho % 4, register rho / 4
            const int r = L.trow[tl] + 4 * (l & 3) + ((l & 15) >> 2);
            const int m = L.member(F::step(ks), F::place(ks), l >> 4);
            if (m < 0 || r >= L.O.size[L.tcls[tl]]) continue;
            const int i = L.O.slot[L.tcls[tl]][r], k = L.O.slot[L.cls(F::step(ks), F::place(ks))][m];
            dst[(((size_t)ks / 2 * F::NT + tl) * 64 + l) * 2 + (ks & 1)] = A[(size_t)k * P2 + i];
          }
    }
  });
}

}  // namespace fmmx
