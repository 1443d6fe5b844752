// m2l_orbit.hip -- M2L of the mixed-precision engine by reflection orbits, on
// the FP16 matrix cores with error compensation.
//
// The offsets (+-dx, +-dy, +-dz) of a target's interaction list (fmm/ijbox.cxx:
// 366-401, kernel/m2l.cxx) share one operator up to diagonal sign matrices
// (OLayout, m2l.h), so the sources of an orbit are combined by a Walsh-Hadamard
// transform first and multiplied once (at most 4 at a time): 63 dense products
// per target instead of 189.  The transformed sources are then carried as FP16
// hi + lo against hi + lo operators (three products, FP32 accumulation), as in
// m2l_split.hip.
#include "orbit.h"

namespace fmmx {

namespace {

// stored position of every float of an orbit box in the padded multipole
// layout (-1: zero), and the partial-sum position of every local slot
template <int P>
struct OTables {
  int16_t src[OConst<P>::BS];
  int16_t pos[P * P];
  constexpr OTables() : src{}, pos{} {
    constexpr OLayout<P> O{};
    using OC = OConst<P>;
    for (int e = 0; e < OC::BS; e++) {
      const bool q = e >= OC::NO * 32;
      const int r = q ? e - OC::NO * 32 : e % 32, s = q ? OC::NO : e / 32;
      const int g = (r % 16) / 4, k = q ? O.qc[r % 4] : 4 * (r / 16) + r % 4, m = 4 * s + g;
      src[e] = m < O.size[k] ? (int16_t)MLayout<P>::at(O.slot[k][m]) : (int16_t)-1;
    }
    for (int k = 0; k < 8; k++)
      for (int i = 0; i < O.size[k]; i++) pos[O.slot[k][i]] = (int16_t)(k * 16 + i);
  }
};
template <int P>
__constant__ OTables<P> c_otab = OTables<P>();

// multipoles of every level in the orbit layout, scaled; the last box of a
// level's range is the zero box.  One thread per stored float (contiguous
// writes, reads within one box).
template <int P>
__global__ __launch_bounds__(256) void k_morder(MSplitLevels S) {
  using OC = OConst<P>;
  const unsigned t = blockIdx.x * 256 + threadIdx.x;
  const long b = t / OC::BS;
  const int e = (int)(t % OC::BS);
  if (b >= S.off[S.nl]) return;
  int k = 0;
  while (k + 1 < S.nl && b >= S.off[k + 1]) k++;
  const int src = c_otab<P>.src[e];
  float v = 0.f;
  if (b != S.off[k + 1] - 1 && src >= 0)
    v = ldexpf(S.M[k][(size_t)(b - S.off[k]) * MLayout<P>::VS + src], orbit_exp(S.mmax[k]));
  reinterpret_cast<float*>(S.Mh[k])[(size_t)(b - S.off[k]) * OC::BS + e] = v;
}

constexpr int ORB_NTH = 64 * ORB_WPG, ORB_TN = 16 * ORB_WPG;

// A workgroup (8 waves) owns 128 targets of one parity class, 16 per wave.
// Per step (octet or quad) a lane reads its words of the product's sources,
// turns them through LDS, transforms and splits them, and the wave multiplies
// the 8 row classes (16 rows each) with their combinations.  One operator in
// LDS (56 KB at P = 10), renewed step by step: once a step's words have
// arrived, the fragments of the step before are replaced by those of one
// product later, copied global -> LDS without registers.
//
// What bounds it (N = 1M, p = 10, levels 2-5): the vector units (transform,
// split, addresses; 6.9e7 instructions, 0.11 ms), the LDS accesses (0.14 ms), the
// L1 accesses of the gather and the MFMAs (0.09 ms) have to overlap, and a
// workgroup's waves move from step to step together: by the counters none is busy
// for half of the launch.
// 0.331 ms for the launch with two workgroups on a CU (128 registers, 76 KB of
// LDS), 0.42 with one (162 registers; holding the fragments of 2 row classes
// instead of 1 spills, 0.357).  Words loaded straight in the product's lane
// order (16 lines per 16 lanes) cost three times the L1 accesses: 0.49 ms,
// 0.40 turned through LDS, in a form with 8 sources per product.  The dense
// form on all 189 offsets (k_m2l_w) takes 0.64 ms; a 120,000-point Plummer
// cloud at p = 8, lmax 7: 0.40 against 0.61.
template <int P>
__global__ __launch_bounds__(ORB_NTH) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_m2l_o(
    M2LLaunch A, const int4* __restrict__ orbtab) {
  M2LLev Q = A.lv[0];
#pragma unroll
  for (int k = 1; k < MAXL + 1; k++)
    if (k < A.nlv && (int)blockIdx.x >= A.lv[k].wg0) Q = A.lv[k];
  using OC = OConst<P>;
  constexpr int NO = OC::NO, QUAD = OC::QUAD, BS = OC::BS, FRO = OC::FRO, FRS = OC::FRS, FRQ = OC::FRQ;
  static_assert(NO >= 1 && NO <= 3);
  constexpr OLayout<P> O{};
  const int lev = Q.lev, nb = Q.nb, nbj = Q.nbj, nsplit = Q.nsplit, gsh = Q.gsh;
  const int* __restrict__ dense_j = Q.dense_j;
  const char* __restrict__ Mb = reinterpret_cast<const char*>(Q.Mh);
  const u32x4* __restrict__ opH = reinterpret_cast<const u32x4*>(Q.opH);
  const int bid = (int)blockIdx.x - Q.wg0, nwg = Q.nwg;
  // one object per step: the compiler then sees the copies into one step's
  // fragments and the reads of another's as independent
  __shared__ u32x4 A0[FRS], A1[NO > 1 ? FRS : 1], A2[NO > 2 ? FRS : 1], Aq[QUAD ? FRQ : 1];
  // per target and axis, the source key's bits at component -3..3 (the sign
  // bit set where that leaves the domain or the group)
  __shared__ uint32_t axk[3][7][ORB_TN];
  __shared__ f32x4 turn[ORB_WPG][64];  // per wave: loaded words on their way to the product's lanes
  __shared__ int s_class, s_start, s_n;
  const int tid = threadIdx.x;
  // tile, class and split of this workgroup: the mapping of k_m2l (XCD b % 8)
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
    const int cnt = Q.cls_cnt[cls0], nt = (cnt + ORB_TN - 1) / ORB_TN;
    s_class = tile < nt ? cls0 : -1;
    s_start = start + tile * ORB_TN;
    s_n = tile < nt ? min(ORB_TN, cnt - tile * ORB_TN) : 0;
  }
  __syncthreads();
  const int cls = __builtin_amdgcn_readfirstlane(s_class), ntile = __builtin_amdgcn_readfirstlane(s_n);
  if (cls < 0) return;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, j = l & 15, kq = l >> 4;
  // The words are loaded with four neighbouring lanes on one target (64
  // contiguous bytes; lane l: target l / 4, group l % 4) and turned through LDS
  // into the product's lanes (target l % 16, group l / 16); the swizzle keeps
  // both sides free of bank conflicts.
  const int tl = l >> 2;
  auto swz = [](int t) { return ((t >> 2) & 1) | (((t >> 3) ^ (t >> 1)) & 1) << 1; };
  const uint32_t kld = (l & 3) * 16u;
  auto lds = [](const f32x4* q_) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const void*)q_; };
  const uint32_t turn_w = lds(&turn[w][tl * 4 + ((l & 3) ^ swz(tl))]), turn_r = lds(&turn[w][j * 4 + (kq ^ swz(j))]);
  const int g = 1 << lev;
  int tord = -1, tx = -16, ty = -16, tz = -16;  // no target: every source out of range
  uint32_t tk = 0u;
  if (w * 16 + j < ntile) {
    tord = (int)Q.ord[s_start + w * 16 + j];
    tk = Q.ikey[tord];
    morton_decode(tk, lev, tx, ty, tz);
  }
  {
    // lane group kq fills the entries kq, kq + 4, ... of its target
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
  f32x4 acc[8];
#pragma unroll
  for (int c = 0; c < 8; c++) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned mypairs = 0;
  const int4* __restrict__ otab = orbtab + cls * NORB;

  // the orbit about to run: byte offsets of its sources' boxes, this lane's
  // words of its first step (entries beyond the orbit's sources are not set)
  uint32_t src[4];
  f32x4 hand[4][2];
  bool any = false;

  // sources of orbit o (-1 where there is none)
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
      uint32_t key = z0 | y0 | x0;
      if (s > 0) {
        const uint32_t mx = (r & 1) ? ~0u : 0u, my = (r & 2) ? ~0u : 0u, mz = (r & 4) ? ~0u : 0u;
        key = ((x1 & mx) | (x0 & ~mx)) | ((y1 & my) | (y0 & ~my)) | ((z1 & mz) | (z0 & ~mz));
      }
      return (int)key >= 0 ? dense_j[key] : -1;
    };
    int v[4];
    v[0] = one(0);
    if (cnt >= 2) v[1] = one(1);
    if (cnt >= 4) v[2] = one(2), v[3] = one(3);
#pragma unroll
    for (int s = 0; s < 4; s++) id[s] = v[s];
  };
  // box offsets of the sources found, and whether the wave has any
  auto take = [&](const int (&id)[4], int cnt) __attribute__((always_inline)) {
    bool a = false;
    auto one = [&](int s) __attribute__((always_inline)) {
      a = a || id[s] >= 0;
      if (id[s] >= 0 && (l & 3) == 0) mypairs++;
      return (uint32_t)(id[s] >= 0 ? id[s] : nbj) * (uint32_t)(BS * 4);
    };
    uint32_t v[4];
    v[0] = one(0);
    if (cnt >= 2) v[1] = one(1);
    if (cnt >= 4) v[2] = one(2), v[3] = one(3);
#pragma unroll
    for (int s = 0; s < 4; s++) src[s] = v[s];
    any = __ballot(a) != 0;
  };
  // unit u of a box (two per octet, one per quad): 4 words per lane
  auto unit = [&](uint32_t box, int u) __attribute__((always_inline)) {
    return *reinterpret_cast<const f32x4*>(Mb + (box + kld + 64u * u));
  };
  // the first step's words of the orbit's sources
  auto first = [&](int cnt) __attribute__((always_inline)) {
    f32x4 v[4][2];
    auto one = [&](int s) __attribute__((always_inline)) {
      v[s][0] = unit(src[s], 0);
      v[s][1] = unit(src[s], 1);
    };
    if (any) {
      one(0);
      if (cnt >= 2) one(1);
      if (cnt >= 4) one(2), one(3);
    }
#pragma unroll
    for (int s = 0; s < 4; s++) hand[s][0] = v[s][0], hand[s][1] = v[s][1];
  };
  auto op_src = [&](int o) __attribute__((always_inline)) -> const u32x4* { return opH + (size_t)(otab[o].w & 0xff) * FRO; };

  __syncthreads();  // axk
  // n fragments of an operator into LDS (global_load_lds: no registers)
  auto copy = [&](const u32x4* src_, u32x4* dst, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < n; e += ORB_NTH)
      __builtin_amdgcn_global_load_lds((const void*)(src_ + e + tid),
                                       (__attribute__((address_space(3))) void*)(dst + e + w * 64), 16, 0, 0);
  };

  // Barrier behind a step, without the wait for all loads that __syncthreads
  // carries: the words loaded during the step and the copies of the step before
  // have arrived, the step's own last n copies (the newest accesses) stay in
  // flight.  They are read NSTEP - 1 >= 2 steps on; with two steps in the very
  // next one, so nothing stays in flight there.
  auto sync = [&](auto nc) __attribute__((always_inline)) {
    constexpr int n = OC::NSTEP == 2 ? 0 : decltype(nc)::value;
    // (the builtin, so that the compiler knows what has arrived)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(n | 7 << 4);  // vmcnt(n) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using NOCT = std::integral_constant<int, FRS / ORB_NTH>;
  using NQUA = std::integral_constant<int, FRQ / ORB_NTH>;
  static_assert(FRS % ORB_NTH == 0 && FRQ % ORB_NTH == 0);

  int o = split;
  if (o < NORB) {
    // every step's fragments but the last's, which step 0 copies
    const u32x4* a = op_src(o);
    if constexpr (NO > 1 || QUAD) copy(a, A0, FRS);
    if constexpr (NO > 2 || (NO == 2 && QUAD)) copy(a + FRS, A1, FRS);
    if constexpr (NO == 3 && QUAD) copy(a + 2 * FRS, A2, FRS);
    int id[4];
    find(o, id);
    const int cnt = 1 << bits3(orb_mask(o));
    take(id, cnt);
    first(cnt);
  }
  sync(std::integral_constant<int, 0>{});

  // the products of one mask D that this split owns
  auto group = [&](auto dc) __attribute__((always_inline)) {
    constexpr int D = decltype(dc)::value, J = bits3(D), NS = 1 << J;
    for (; o < orb_start(D + 1); o += nsplit) {
      const int on = o + nsplit;
      const bool more = on < NORB;
      const u32x4* acur = op_src(o);
      const u32x4* anext = op_src(more ? on : o);
      int id[4];
      int cntn = 0;
      if (more) {
        cntn = 1 << bits3(orb_mask(on));
        find(on, id);
      }
      const bool run = any;
      f32x4 ld[NS][2];  // words in flight or loaded
      uint32_t box[NS];
#pragma unroll
      for (int s = 0; s < NS; s++) {
        box[s] = src[s];
        ld[s][0] = hand[s][0], ld[s][1] = hand[s][1];
      }
      // the loaded words of unit h into the product's lanes, one source after
      // the other (a wave's LDS accesses stay in order).  Store, load and wait
      // in one block: the compiler would hold a load from this array back until
      // every copy into LDS has landed.
      auto turned = [&](float(&raw)[NS][4], const f32x4(&ld_)[NS][2], int h) __attribute__((always_inline)) {
        if constexpr (NS == 1) {
          f32x4 u = ld_[0][h];
          asm volatile("ds_write_b128 %1, %0\n\tds_read_b128 %0, %2\n\ts_waitcnt lgkmcnt(0)"
                       : "+v"(u)
                       : "v"(turn_w), "v"(turn_r)
                       : "memory");
#pragma unroll
          for (int t = 0; t < 4; t++) raw[0][t] = u[t];
        } else {
#pragma unroll
          for (int q = 0; q < NS; q += 2) {
            f32x4 u = ld_[q][h], v = ld_[q + 1][h];
            asm volatile("ds_write_b128 %2, %0\n\tds_read_b128 %0, %3\n\tds_write_b128 %2, %1\n\t"
                         "ds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                         : "+v"(u), "+v"(v)
                         : "v"(turn_w), "v"(turn_r)
                         : "memory");
#pragma unroll
            for (int t = 0; t < 4; t++) raw[q][t] = u[t], raw[q + 1][t] = v[t];
          }
        }
      };
      // the last step's words are in registers: the next orbit's first step
      auto next_orbit = [&]() __attribute__((always_inline)) {
        if (more) take(id, cntn);
        else any = false;
        first(cntn);
      };
      // the 8 row classes of a step: a class's fragments, then its products
      // (three in a row on one accumulator: the SIMD's other waves fill in)
      auto products = [&](const u32x4* Ab, const u32x4(&bh)[NS], const u32x4(&bl)[NS], auto qc) __attribute__((always_inline)) {
        constexpr bool QS = decltype(qc)::value;
#pragma unroll
        for (int c = 0; c < 8; c++) {
          const h8 hi = __builtin_bit_cast(h8, bh[sub_rank(D, c & D)]), lo = __builtin_bit_cast(h8, bl[sub_rank(D, c & D)]);
          const h8 ah = __builtin_bit_cast(h8, Ab[(QS ? c : 2 * c) * 64]);
          h8 al;
          if constexpr (!QS) al = __builtin_bit_cast(h8, Ab[(2 * c + 1) * 64]);
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, hi, acc[c], 0, 0, 0);
          if constexpr (!QS) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, hi, acc[c], 0, 0, 0);
          acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, lo, acc[c], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      };
      auto step = [&](auto sc, const u32x4* Ab) __attribute__((always_inline)) {
        constexpr int s = decltype(sc)::value;
        // the fragments of the step before this one are free
        auto renew = [&]() __attribute__((always_inline)) {
          if constexpr (s == 0) {
            if constexpr (QUAD) copy(acur + NO * FRS, Aq, FRQ);
            else if constexpr (NO == 3) copy(acur + 2 * FRS, A2, FRS);
            else if constexpr (NO == 2) copy(acur + FRS, A1, FRS);
          } else if constexpr (s == 1) {
            copy(anext, A0, FRS);
          } else {
            copy(anext + FRS, A1, FRS);
          }
        };
        if (run) {
          u32x4 bh[NS], bl[NS];
          // words 4 h .. 4 h + 3: transform, split, and their registers take
          // the next step's words
#pragma unroll
          for (int h = 0; h < 2; h++) {
            float raw[NS][4];
            turned(raw, ld, h);
#pragma unroll
            for (int t = 0; t < 4; t++) wht<J>(raw, t);
#pragma unroll
            for (int c = 0; c < NS; c++)
#pragma unroll
              for (int a = 2 * h; a < 2 * h + 2; a++) {
                const float e0 = raw[c ^ sub_rank(D, (2 * a) & D)][2 * a - 4 * h];
                const float e1 = raw[c ^ sub_rank(D, (2 * a + 1) & D)][2 * a + 1 - 4 * h];
                bh[c][a] = hi_pair(e0, e1);
                bl[c][a] = lo_pair(e0, e1, bh[c][a]);
              }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (s + 1 < NO) {
#pragma unroll
              for (int q = 0; q < NS; q++) ld[q][h] = unit(box[q], 2 * s + 2 + h);
            } else if (QUAD && h == 0) {
              // (the quad's one unit follows the last octet's two)
#pragma unroll
              for (int q = 0; q < NS; q++) ld[q][h] = unit(box[q], 2 * s + 2 + h);
            } else if (!QUAD && h == 1) {
              next_orbit();
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          renew();
          __builtin_amdgcn_sched_barrier(0);
          products(Ab + l, bh, bl, std::false_type{});
        } else {
          if constexpr (!QUAD && s + 1 == NO) next_orbit();
          renew();
        }
        if constexpr (s == 0 && QUAD) sync(NQUA{});
        else sync(NOCT{});
      };
      step(std::integral_constant<int, 0>{}, A0);
      if constexpr (NO > 1) step(std::integral_constant<int, 1>{}, A1);
      if constexpr (NO > 2) step(std::integral_constant<int, 2>{}, A2);
      if constexpr (QUAD) {
        auto renew = [&]() __attribute__((always_inline)) {
          copy(anext + (NO - 1) * FRS, NO == 1 ? A0 : NO == 2 ? A1 : A2, FRS);
        };
        if (run) {
          u32x4 bh[NS], bl[NS];
          float raw[NS][4];
          turned(raw, ld, 0);
#pragma unroll
          for (int t = 0; t < 4; t++) wht<J>(raw, t);
#pragma unroll
          for (int c = 0; c < NS; c++)
#pragma unroll
            for (int a = 0; a < 2; a++) {
              const float e0 = raw[c ^ sub_rank(D, O.qc[2 * a] & D)][2 * a];
              const float e1 = raw[c ^ sub_rank(D, O.qc[2 * a + 1] & D)][2 * a + 1];
              bh[c][a] = bh[c][2 + a] = hi_pair(e0, e1);
              bl[c][a] = lo_pair(e0, e1, bh[c][a]);
              bl[c][2 + a] = 0u;
            }
          __builtin_amdgcn_sched_barrier(0);
          next_orbit();
          renew();
          __builtin_amdgcn_sched_barrier(0);
          products(Aq + l, bh, bl, std::true_type{});
        } else {
          next_orbit();
          renew();
        }
        sync(NOCT{});
      }
    }
  };
  group(std::integral_constant<int, 0>{});
  group(std::integral_constant<int, 1>{});
  group(std::integral_constant<int, 2>{});
  group(std::integral_constant<int, 3>{});
  group(std::integral_constant<int, 4>{});
  group(std::integral_constant<int, 5>{});
  group(std::integral_constant<int, 6>{});

  const int oexp = -(orbit_exp(Q.mmax) + Q.sa_e);
  if (tord >= 0) {
    f32x4* dst = reinterpret_cast<f32x4*>(Q.part + ((size_t)split * nb + tord) * OC::ROWS + 4 * kq);
#pragma unroll
    for (int c = 0; c < 8; c++)
      dst[4 * c] = f32x4{ldexpf(acc[c][0], oexp), ldexpf(acc[c][1], oexp), ldexpf(acc[c][2], oexp), ldexpf(acc[c][3], oexp)};
  }
  if (mypairs) atomicAdd(Q.npairs, (unsigned long long)mypairs);
}

// the partial sums of every level into the locals, splits in fixed order
struct OReduce {
  const float* part[MAXL + 1];
  float* L[MAXL + 1];
  unsigned off[MAXL + 2];
  int nsplit[MAXL + 1], nb[MAXL + 1], init[MAXL + 1];
  int nl;
};
template <int P>
__global__ __launch_bounds__(256) void k_orbit_reduce(OReduce R) {
  constexpr int P2 = P * P, ROWS = OConst<P>::ROWS;
  const unsigned t = blockIdx.x * 256 + threadIdx.x, b = t / P2;
  const int i = (int)(t % P2);
  if (b >= R.off[R.nl]) return;
  int k = 0;
  while (k + 1 < R.nl && b >= R.off[k + 1]) k++;
  const unsigned bl = b - R.off[k];
  const float* p = R.part[k] + (size_t)bl * ROWS + c_otab<P>.pos[i];
  float* L = R.L[k] + (size_t)bl * P2 + i;
  float s = R.init[k] ? 0.f : *L;
  for (int q = 0; q < R.nsplit[k]; q++) s += p[(size_t)q * R.nb[k] * ROWS];
  *L = s;
}

template <typename F>
int dispatch_orbit_p(int p, F&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(6) FMMX_CASE(7) FMMX_CASE(8) FMMX_CASE(9) FMMX_CASE(10)
#undef FMMX_CASE
  }
  return fail(FMMX_EUNSUPPORTED, "the orbit M2L covers p = 6..10");
}

}  // namespace

int launch_morder(int p, const MSplitLevels& S, hipStream_t stream) {
  return dispatch_orbit_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    const long n = S.off[S.nl] * OConst<P>::BS;
    if (n >= (1L << 32)) return fail(FMMX_EUNSUPPORTED, "too many boxes for the orbit M2L");
    k_morder<P><<<(int)((n + 255) / 256), 256, 0, stream>>>(S);
    return FMMX_OK;
  });
}

int launch_m2l_orbit(int p, const M2LLaunch& A, int nwg, const int4* orbtab, hipStream_t stream) {
  return dispatch_orbit_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    k_m2l_o<P><<<nwg, ORB_NTH, 0, stream>>>(A, orbtab);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "orbit M2L launch failed");
  });
}

int launch_orbit_reduce(int p, const M2LLaunch& A, hipStream_t stream) {
  return dispatch_orbit_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    OReduce R{};
    for (int k = 0; k < A.nlv; k++) {
      const M2LLev& d = A.lv[k];
      R.part[k] = d.part;
      R.L[k] = d.L;
      R.nsplit[k] = d.nsplit;
      R.nb[k] = d.nb;
      R.init[k] = d.init;
      R.off[k + 1] = R.off[k] + (unsigned)d.nb;
      R.nl++;
    }
    const long n = (long)R.off[R.nl] * P * P;
    if (n >= (1L << 32)) return fail(FMMX_EUNSUPPORTED, "too many boxes for the orbit M2L");
    k_orbit_reduce<P><<<(int)((n + 255) / 256), 256, 0, stream>>>(R);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "orbit M2L reduction launch failed");
  });
}

}  // namespace fmmx
