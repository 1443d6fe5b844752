// m2l_orbit_fp64.hip -- M2L of the FP64 engine by reflection orbits on the FP64
// matrix cores (Laplace, EXACT, p = 6..12): 63 products per target instead of
// 189, with the sums over an orbit's sources and all products in FP64.
#include "mfma.h"
#include "orbit.h"

namespace fmmx {

namespace {

typedef double d2 __attribute__((ext_vector_type(2)));

template <int P>
struct FTables {
  using F = FConst<P>;
  int16_t src[F::BS];
  int16_t pos[P * P];
  constexpr FTables() : src{}, pos{} {
    constexpr GLayout<P> L{};
    for (int e = 0; e < F::BS; e++) {
      const int ks = e / 8 * 2 + (e & 1), g = (e & 7) >> 1, s = F::step(ks), t = F::place(ks);
      const int m = L.member(s, t, g);
      src[e] = m < 0 ? (int16_t)-1 : (int16_t)MLayout<P>::at(L.O.slot[L.cls(s, t)][m]);
    }
    for (int tl = 0; tl < F::NT; tl++)
      for (int r = 0; r < 16; r++)
        if (L.trow[tl] + r < L.O.size[L.tcls[tl]]) pos[L.O.slot[L.tcls[tl]][L.trow[tl] + r]] = (int16_t)(tl * 16 + r);
  }
};
template <int P>
__constant__ FTables<P> c_ftab = FTables<P>();

// multipoles of every level in the stored layout, and a zero box after each level's
template <int P>
__global__ __launch_bounds__(256) void k_forder(MSplitLevels S) {
  using F = FConst<P>;
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  const long b = (long)(t / F::BS);
  const int e = (int)(t % F::BS);
  if (b >= S.off[S.nl]) return;
  int k = 0;
  while (k + 1 < S.nl && b >= S.off[k + 1]) k++;
  const int src = c_ftab<P>.src[e];
  double v = 0.0;
  if (b != S.off[k + 1] - 1 && src >= 0)
    v = reinterpret_cast<const double*>(S.M[k])[(size_t)(b - S.off[k]) * MLayout<P>::VS + src];
  reinterpret_cast<double*>(S.Mh[k])[(size_t)(b - S.off[k]) * F::BS + e] = v;
}

constexpr int F64_NTH = 64 * ORB_WPG, F64_TN = 16 * ORB_WPG;

// 16 targets per wave: lanes of target l % 16 and k-group l / 16 of
// v_mfma_f64_16x16x4, words (two k-steps, 16 bytes) loaded with four lanes on
// one target and turned through LDS.  Operator fragments go through two LDS
// buffers of eight k-steps, copied one step ahead; one barrier per step.
//
// What bounds it: the FP64 matrix cores (64 cycles per MFMA at the 78.6
// TFLOP/s of the card; busy for 49 % of the launch below by the counters, the LDS
// for 16 %) and the steps' barriers, on row tiles padded to 16: 224 MFMAs per
// product and 16 targets at p = 10, where 100 x 100 are 156.  N = 250k, p = 10,
// lmax 4 (640,584 pairs): 0.228 ms for the launch of all levels, beside the near
// field; 0.89 + 1.34 ms as 189 products per target on the vector units with
// operands re-read from LDS, which this replaces.
template <int P>
__global__ __launch_bounds__(F64_NTH) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_m2l_of(
    M2LLaunch A, const int4* __restrict__ orbtab) {
  M2LLev Q = A.lv[0];
#pragma unroll
  for (int k = 1; k < MAXL + 1; k++)
    if (k < A.nlv && (int)blockIdx.x >= A.lv[k].wg0) Q = A.lv[k];
  using F = FConst<P>;
  constexpr int NT = F::NT, CH = F::CH;
  constexpr GLayout<P> L{};
  const int lev = Q.lev, nb = Q.nb, nbj = Q.nbj, nsplit = Q.nsplit, gsh = Q.gsh;
  const int* __restrict__ dense_j = Q.dense_j;
  const char* __restrict__ Mb = reinterpret_cast<const char*>(Q.Mh);
  const u32x4* __restrict__ opH = reinterpret_cast<const u32x4*>(Q.opH);
  const int bid = (int)blockIdx.x - Q.wg0, nwg = Q.nwg;
  __shared__ u32x4 As[2 * CH];
  __shared__ uint32_t axk[3][7][F64_TN];   // source key bits per target, axis and component
  __shared__ f32x4 turn[ORB_WPG][64];
  __shared__ int s_class, s_start, s_n;
  const int tid = threadIdx.x;
  int cls0, split, tile;
  if (Q.region) {
    const int xcd = bid & 7, item = bid >> 3, tpr = (nwg >> 6) / nsplit;
    cls0 = item & 7;
    split = (item >> 3) % nsplit;
    tile = xcd * tpr + (item >> 3) / nsplit;
  } else {
    const int item = bid >> 3, tpc = (nwg >> 3) / nsplit;
    cls0 = bid & 7;
    split = item / tpc;
    tile = item % tpc;
  }
  if (tid == 0) {
    int start = 0;
    for (int c = 0; c < cls0; c++) start += Q.cls_cnt[c];
    const int cnt = Q.cls_cnt[cls0], nt = (cnt + F64_TN - 1) / F64_TN;
    s_class = tile < nt ? cls0 : -1;
    s_start = start + tile * F64_TN;
    s_n = tile < nt ? min(F64_TN, cnt - tile * F64_TN) : 0;
  }
  __syncthreads();
  const int cls = __builtin_amdgcn_readfirstlane(s_class), ntile = __builtin_amdgcn_readfirstlane(s_n);
  if (cls < 0) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, j = l & 15, kq = l >> 4, tl = l >> 2;
  auto swz = [](int t) { return ((t >> 2) & 1) | (((t >> 3) ^ (t >> 1)) & 1) << 1; };
  const uint32_t kld = (l & 3) * 16u;
  auto lds = [](const void* q_) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)q_; };
  const uint32_t turn_w = lds(&turn[w][tl * 4 + ((l & 3) ^ swz(tl))]), turn_r = lds(&turn[w][j * 4 + (kq ^ swz(j))]);
  const uint32_t as_base = __builtin_amdgcn_readfirstlane(lds(&As[0]));
  const int g = 1 << lev;
  int tord = -1;
  {
    int tx = -16, ty = -16, tz = -16;  // no target: every source out of range
    uint32_t tk = 0u;
    if (w * 16 + j < ntile) {
      tord = (int)Q.ord[s_start + w * 16 + j];
      tk = Q.ikey[tord];
      morton_decode(tk, lev, tx, ty, tz);
    }
    const uint32_t MY = 0x49249249u & ((1u << (3 * lev)) - 1u);
    for (int e = kq; e < 21; e += 4) {
      const int ax = e / 7, d = e % 7 - 3, t = ax == 0 ? tx : ax == 1 ? ty : tz, jj = t - d;
      const int sh = ax == 0 ? 1 : ax == 1 ? 0 : 2;
      const uint32_t M = MY << sh, dil = dil3(abs(d)) << sh;
      const bool ok = (unsigned)jj < (unsigned)g && (gsh < 0 || !((jj ^ t) >> gsh));
      const uint32_t k = d >= 0 ? ((tk & M) - dil) & M : ((tk | ~M) + dil) & M;
      axk[ax][d + 3][w * 16 + j] = ok ? k : 0x80000000u;
    }
  }
  f64x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) acc[t] = Mfma<double>::zero();
  unsigned mypairs = 0;
  const int4* __restrict__ otab = orbtab + cls * NORB;
  uint32_t src[4];  // boxes of the product about to run, in 64-byte units
  f32x4 hand[4];    // this lane's first word of it
  bool any = false;

  auto find = [&](int o, int (&id)[4]) __attribute__((always_inline)) {
    const int4 of = otab[o];
    const int cnt = 1 << bits3(orb_mask(o));
    const uint32_t subs = (uint32_t)of.w >> 8;
    const int t = w * 16 + tl;
    const uint32_t x0 = axk[0][3 + of.x][t], x1 = axk[0][3 - of.x][t];
    const uint32_t y0 = axk[1][3 + of.y][t], y1 = axk[1][3 - of.y][t];
    const uint32_t z0 = axk[2][3 + of.z][t], z1 = axk[2][3 - of.z][t];
    auto one = [&](int s) __attribute__((always_inline)) {
      const int r = (subs >> (3 * s)) & 7;
      const uint32_t mx = (r & 1) ? ~0u : 0u, my = (r & 2) ? ~0u : 0u, mz = (r & 4) ? ~0u : 0u;
      const uint32_t key = ((x1 & mx) | (x0 & ~mx)) | ((y1 & my) | (y0 & ~my)) | ((z1 & mz) | (z0 & ~mz));
      return (int)key >= 0 ? dense_j[key] : -1;
    };
    int v[4];
    v[0] = one(0);
    if (cnt >= 2) v[1] = one(1);
    if (cnt >= 4) v[2] = one(2), v[3] = one(3);
#pragma unroll
    for (int s = 0; s < 4; s++) id[s] = v[s];
  };
  auto unit = [&](uint32_t box, int u) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(Mb + ((size_t)(box + (uint32_t)u) * 64 + kld));
  };
  // the sources found for the next product, and its first word
  auto take = [&](const int (&id)[4], int cnt) __attribute__((always_inline)) {
    bool a = false;
    auto one = [&](int s) __attribute__((always_inline)) {
      a = a || id[s] >= 0;
      if (id[s] >= 0 && (l & 3) == 0) mypairs++;
      return (uint32_t)(id[s] >= 0 ? id[s] : nbj) * (uint32_t)F::NU;
    };
    uint32_t v[4];
    v[0] = one(0);
    if (cnt >= 2) v[1] = one(1);
    if (cnt >= 4) v[2] = one(2), v[3] = one(3);
#pragma unroll
    for (int s = 0; s < 4; s++) src[s] = v[s];
    any = __ballot(a) != 0;
  };
  auto first = [&](int cnt) __attribute__((always_inline)) {
    f32x4 v[4];
    if (any) {
      v[0] = unit(src[0], 0);
      if (cnt >= 2) v[1] = unit(src[1], 0);
      if (cnt >= 4) v[2] = unit(src[2], 0), v[3] = unit(src[3], 0);
    }
#pragma unroll
    for (int s = 0; s < 4; s++) hand[s] = v[s];
  };
  // n fragments of a step into LDS buffer b; sync() waits for them
  auto copy = [&](const u32x4* from, int b, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < CH; e += F64_NTH)
      if (e + w * 64 < n) lds_copy16(as_base + (b * CH + e + w * 64) * 16, from + e + tid);
  };
  auto op_src = [&](int o) __attribute__((always_inline)) -> const u32x4* { return opH + (size_t)(otab[o].w & 0xff) * F::FRO; };
  // every access of the step behind has arrived in every wave
  auto sync = [&]() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  sync();  // axk
  int buf = 0, o = split;
  if (o < NORB) {
    copy(op_src(o), 0, CH);
    int id[4];
    find(o, id);
    const int cnt = 1 << bits3(orb_mask(o));
    take(id, cnt);
    first(cnt);
  }
  sync();

  // the products of one mask D that this split owns
  auto group = [&](auto dc) __attribute__((always_inline)) {
    constexpr int D = decltype(dc)::value, J = bits3(D), NS = 1 << J;
    for (; o < orb_start(D + 1); o += nsplit) {
      const int on = o + nsplit;
      const bool more = on < NORB;
      const u32x4 *acur = op_src(o), *anext = op_src(more ? on : o);
      int id[4];
      int cntn = 0;
      if (more) {
        cntn = 1 << bits3(orb_mask(on));
        find(on, id);
      }
      const bool run = any;
      f32x4 ld[NS];
      uint32_t box[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) box[s] = src[s], ld[s] = hand[s];
      auto next_product = [&]() __attribute__((always_inline)) {
        if (more) take(id, cntn);
        else any = false;
        first(cntn);
      };
      auto turned = [&](double(&raw)[NS][2]) __attribute__((always_inline)) {
        if constexpr (NS == 1) {
          f32x4 u = ld[0];
          asm volatile("ds_write_b128 %1, %0\n\tds_read_b128 %0, %2\n\ts_waitcnt lgkmcnt(0)"
                       : "+v"(u)
                       : "v"(turn_w), "v"(turn_r)
                       : "memory");
          const d2 a = __builtin_bit_cast(d2, u);
          raw[0][0] = a[0], raw[0][1] = a[1];
        } else {
#pragma unroll
          for (int q = 0; q < NS; q += 2) {
            f32x4 u = ld[q], v = ld[q + 1];
            asm volatile("ds_write_b128 %2, %0\n\tds_read_b128 %0, %3\n\tds_write_b128 %2, %1\n\t"
                         "ds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                         : "+v"(u), "+v"(v)
                         : "v"(turn_w), "v"(turn_r)
                         : "memory");
            const d2 a = __builtin_bit_cast(d2, u), b = __builtin_bit_cast(d2, v);
            raw[q][0] = a[0], raw[q][1] = a[1];
            raw[q + 1][0] = b[0], raw[q + 1][1] = b[1];
          }
        }
      };
      // step s of NW words; XT: the last octet of the larger classes; LAST: the
      // product's last step
      auto step = [&](int s, auto xt, auto lc) __attribute__((always_inline)) {
        constexpr bool XT = decltype(xt)::value, LAST = decltype(lc)::value;
        constexpr int NW = XT ? F::NKX / 2 : 4;
        auto ahead = [&]() __attribute__((always_inline)) {
          if constexpr (LAST) copy(anext, buf ^ 1, CH);
          else copy(acur + (size_t)(s + 1) * CH, buf ^ 1, F::XTRA && s + 1 == F::NO ? F::CHX : CH);
        };
        if (!run) {
          ahead();
          if constexpr (LAST) next_product();
          return;
        }
        const d2* Ab = reinterpret_cast<const d2*>(As + buf * CH) + l;
#pragma unroll
        for (int u = 0; u < NW; u++) {
          double raw[NS][2];
          turned(raw);
#pragma unroll
          for (int b = 0; b < J; b++)
#pragma unroll
            for (int q = 0; q < NS; q++)
              if (!(q & (1 << b)))
#pragma unroll
                for (int h = 0; h < 2; h++) {
                  const double x = raw[q][h], y = raw[q | (1 << b)][h];
                  raw[q][h] = x + y;
                  raw[q | (1 << b)][h] = x - y;
                }
          __builtin_amdgcn_sched_barrier(0);
          if (u + 1 < NW || !LAST) {
#pragma unroll
            for (int q = 0; q < NS; q++) ld[q] = unit(box[q], 4 * s + u + 1);
          } else {
            next_product();
          }
          if (u == 0) ahead();  // behind the words: their wait covers no copy yet
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int t = 0; t < NT; t++) {
            const d2 f = Ab[(u * NT + t) * 64];
#pragma unroll
            for (int h = 0; h < 2; h++) {
              const int kc = XT ? L.qc[(2 * u + h) & 3] : 2 * u + h;
              const int c = sub_rank(D, (L.tcls[t] ^ kc) & D);
              acc[t] = Mfma<double>::fma(f[h], raw[c][h], acc[t]);
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      };
#pragma unroll 1
      for (int s = 0; s < F::NSTEP - 1; s++) {
        step(s, std::false_type{}, std::false_type{});
        sync();
        buf ^= 1;
      }
      step(F::NSTEP - 1, std::integral_constant<bool, F::XTRA != 0>{}, std::true_type{});
      sync();
      buf ^= 1;
    }
  };
  group(std::integral_constant<int, 0>{});
  group(std::integral_constant<int, 1>{});
  group(std::integral_constant<int, 2>{});
  group(std::integral_constant<int, 3>{});
  group(std::integral_constant<int, 4>{});
  group(std::integral_constant<int, 5>{});
  group(std::integral_constant<int, 6>{});

  // the operators' rows are ordered so that a lane holds four rows in turn
  if (tord >= 0) {
    f64x4* dst = reinterpret_cast<f64x4*>(reinterpret_cast<double*>(Q.part) + ((size_t)split * nb + tord) * F::ROWS + 4 * kq);
#pragma unroll
    for (int t = 0; t < NT; t++) dst[4 * t] = acc[t];
  }
  if (mypairs) atomicAdd(Q.npairs, (unsigned long long)mypairs);
}

// the partial sums of every level into the locals, splits in fixed order
struct FReduce {
  const double* part[MAXL + 1];
  double* L[MAXL + 1];
  unsigned off[MAXL + 2];
  int nsplit[MAXL + 1], nb[MAXL + 1], init[MAXL + 1];
  int nl;
};
template <int P>
__global__ __launch_bounds__(256) void k_f64_reduce(FReduce R) {
  using F = FConst<P>;
  constexpr int N = P * P;
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  const unsigned b = (unsigned)(t / N);
  const int i = (int)(t % N);
  if (t >= (size_t)R.off[R.nl] * N) return;
  int k = 0;
  while (k + 1 < R.nl && b >= R.off[k + 1]) k++;
  const unsigned bl = b - R.off[k];
  const double* p = R.part[k] + (size_t)bl * F::ROWS + c_ftab<P>.pos[i];
  double* L = R.L[k] + (size_t)bl * N + i;
  double s = R.init[k] ? 0.0 : *L;
  for (int q = 0; q < R.nsplit[k]; q++) s += p[(size_t)q * R.nb[k] * F::ROWS];
  *L = s;
}

template <typename G>
int dispatch_f64(int p, G&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(6) FMMX_CASE(7) FMMX_CASE(8) FMMX_CASE(9) FMMX_CASE(10) FMMX_CASE(11) FMMX_CASE(12)
#undef FMMX_CASE
  }
  return fail(FMMX_EUNSUPPORTED, "order without an FP64 orbit M2L");
}

}  // namespace

// reorders the multipoles, runs the launch (between the events, if given) and
// adds its partial sums to the locals
int launch_m2l_orbit_f64(int p, const MSplitLevels& S, const M2LLaunch& A, int nwg, const int4* orbtab, hipEvent_t e0,
                         hipEvent_t e1, hipStream_t stream) {
  return dispatch_f64(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    using F = FConst<P>;
    const long n = S.off[S.nl] * F::BS;
    k_forder<P><<<(int)((n + 255) / 256), 256, 0, stream>>>(S);
    if (e0) FMMX_HIP(hipEventRecord(e0, stream));
    k_m2l_of<P><<<nwg, F64_NTH, 0, stream>>>(A, orbtab);
    if (e1) FMMX_HIP(hipEventRecord(e1, stream));
    FReduce R{};
    for (int k = 0; k < A.nlv; k++) {
      const M2LLev& d = A.lv[k];
      R.part[k] = reinterpret_cast<const double*>(d.part);
      R.L[k] = reinterpret_cast<double*>(d.L);
      R.nsplit[k] = d.nsplit;
      R.nb[k] = d.nb;
      R.init[k] = d.init;
      R.off[k + 1] = R.off[k] + (unsigned)d.nb;
      R.nl++;
    }
    const long nr = (long)R.off[R.nl] * P * P;
    k_f64_reduce<P><<<(int)((nr + 255) / 256), 256, 0, stream>>>(R);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "FP64 orbit M2L launch failed");
  });
}

}  // namespace fmmx
