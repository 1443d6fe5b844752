// m2l_orbit_gen.hip -- M2L by reflection orbits of the FP32 engine's Helmholtz
// kernel (split expansions of two parts, row classes of up to 21 slots at
// p = 12), on the FP16 matrix cores with error compensation (hi/lo operands,
// three products, FP32 accumulation).
#include "orbit.h"

namespace fmmx {

namespace {

template <int P>
struct GTables {
  using G = GConst<P>;
  int16_t src[G::BS];
  int16_t pos[G::PARTS * G::P2];
  constexpr GTables() : src{}, pos{} {
    constexpr GLayout<P> L{};
    for (int e = 0; e < G::BS; e++) {
      const int part = e / G::PBS, r = e % G::PBS, s = r / 32, h = (r % 32) / 16, g = (r % 16) / 4, t = 4 * h + r % 4;
      const int m = L.member(s, t, g);
      src[e] = m < 0 ? (int16_t)-1 : (int16_t)(part * MLayout<P>::VS + MLayout<P>::at(L.O.slot[L.cls(s, t)][m]));
    }
    for (int part = 0; part < G::PARTS; part++)
      for (int tl = 0; tl < G::NT; tl++)
        for (int r = 0; r < 16; r++)
          if (L.trow[tl] + r < L.O.size[L.tcls[tl]])
            pos[part * G::P2 + L.O.slot[L.tcls[tl]][L.trow[tl] + r]] = (int16_t)((part * G::NT + tl) * 16 + r);
  }
};
template <int P>
__constant__ GTables<P> c_gtab = GTables<P>();

// scale word of box b of the flattened range, in level k
__device__ __forceinline__ unsigned* scale_word(const MSplitLevels& S, int k, long b) {
  return S.mmax[k] + (S.ng > 1 ? S.key[k][b - S.off[k]] >> (3 * S.gs[k]) : 0u);
}

// largest |multipole| of every level and group (float bits; zeroed before), 8 floats
// per thread: a box is PARTS padded vectors, whose pads are zero.  Waves and
// workgroups within one scale word reduce before the global atomic.
template <int P>
__global__ __launch_bounds__(256) void k_gmax(MSplitLevels S) {
  constexpr int N8 = GConst<P>::PARTS * MLayout<P>::VS / 8;
  const long t = (long)blockIdx.x * 256 + threadIdx.x, b = t / N8;
  __shared__ unsigned smax;
  __shared__ unsigned* sword;
  int k = 0;
  while (k + 1 < S.nl && b >= S.off[k + 1]) k++;
  float mx = 0.f;
  unsigned* word = S.mmax[k];
  if (b < S.off[S.nl] && b != S.off[k + 1] - 1) {
    const f32x4* m = reinterpret_cast<const f32x4*>(S.M[k]) + ((size_t)(b - S.off[k]) * N8 + t % N8) * 2;
    const f32x4 u = m[0], v = m[1];
#pragma unroll
    for (int e = 0; e < 4; e++) mx = fmaxf(mx, fmaxf(fabsf(u[e]), fabsf(v[e])));
    word = scale_word(S, k, b);
  }
  if (threadIdx.x == 0) {
    smax = 0u;
    sword = word;
  }
  __syncthreads();
  unsigned* const mine = sword;
  if (__ballot(word != mine) == 0) {
    for (int d = 32; d > 0; d >>= 1) mx = fmaxf(mx, __shfl_xor(mx, d));
    if ((threadIdx.x & 63) == 0 && mx > 0.f) atomicMax(&smax, __float_as_uint(mx));
  } else if (mx > 0.f) {
    atomicMax(word == mine ? &smax : word, __float_as_uint(mx));
  }
  __syncthreads();
  if (threadIdx.x == 0 && smax) atomicMax(mine, smax);
}
__global__ __launch_bounds__(256) void k_gzero(MSplitLevels S) {
  const unsigned t = blockIdx.x * 256 + threadIdx.x;
  if (t < (unsigned)(S.nl * S.ng)) S.mmax[t / S.ng][t % S.ng] = 0u;
}

// multipoles of every level in the stored layout, scaled (as k_morder)
template <int P>
__global__ __launch_bounds__(256) void k_gorder(MSplitLevels S) {
  using G = GConst<P>;
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  const long b = (long)(t / G::BS);
  const int e = (int)(t % G::BS);
  if (b >= S.off[S.nl]) return;
  int k = 0;
  while (k + 1 < S.nl && b >= S.off[k + 1]) k++;
  const int src = c_gtab<P>.src[e];
  float v = 0.f;
  if (b != S.off[k + 1] - 1 && src >= 0)
    v = ldexpf(S.M[k][(size_t)(b - S.off[k]) * G::PARTS * MLayout<P>::VS + src], orbit_exp(scale_word(S, k, b)));
  reinterpret_cast<float*>(S.Mh[k])[(size_t)(b - S.off[k]) * G::BS + e] = v;
}

constexpr int GEN_NTH = 64 * ORB_WPG, GEN_TN = 16 * ORB_WPG;

// As k_m2l_o: 16 targets per wave, lanes of target l % 16 and lane group l / 16,
// words loaded with four lanes on one target and turned through LDS.  Per step
// both parts are transformed in turn and multiplied with the step's C and S
// fragments: Re += C R - S I, Im += S R + C I.  Two LDS buffers of one step's
// fragments (48 KB at P = 12): the next step's are copied while this one's
// products run (144 MFMAs per wave), one barrier per step.
//
// What bounds it: latency.  By the counters (sphere of 1M points, p = 12) the
// matrix cores are busy for 29 % of the launch, the LDS for 30 %, the vector units
// for 15 %: one workgroup per CU, whose two waves per SIMD move behind a barrier per
// step, and for 27 % of the CU time none.  Levels 2-6 there (1.12M pairs): 1.35 ms
// for the launch, 8.87 ms as FP32 MFMA products of 288 x 288
// operators per offset, which this replaces (1.64 ms with each tile's fragments
// waited for before its products).  Taking products without any source in the
// workgroup off its list beforehand gained nothing: few are empty for 128
// targets.
template <int P>
__global__ __launch_bounds__(GEN_NTH) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_m2l_og(
    M2LLaunch A, const int4* __restrict__ orbtab) {
  M2LLev Q = A.lv[0];
#pragma unroll
  for (int k = 1; k < MAXL + 1; k++)
    if (k < A.nlv && (int)blockIdx.x >= A.lv[k].wg0) Q = A.lv[k];
  using G = GConst<P>;
  constexpr int NSTEP = G::NSTEP, NT = G::NT, PARTS = G::PARTS, CH = G::CH, FRO = G::FRO;
  constexpr GLayout<P> L{};
  const int lev = Q.lev, nb = Q.nb, nbj = Q.nbj, nsplit = Q.nsplit, gsh = Q.gsh;
  const int* __restrict__ dense_j = Q.dense_j;
  const char* __restrict__ Mb = reinterpret_cast<const char*>(Q.Mh);
  const u32x4* __restrict__ opH = reinterpret_cast<const u32x4*>(Q.opH);
  const int bid = (int)blockIdx.x - Q.wg0, nwg = Q.nwg;
  __shared__ u32x4 As[2 * CH];
  __shared__ uint32_t axk[3][7][GEN_TN];   // source key bits per target, axis and component (k_m2l_o)
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
    const int cnt = Q.cls_cnt[cls0], nt = (cnt + GEN_TN - 1) / GEN_TN;
    s_class = tile < nt ? cls0 : -1;
    s_start = start + tile * GEN_TN;
    s_n = tile < nt ? min(GEN_TN, cnt - tile * GEN_TN) : 0;
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
  static_assert(CH % GEN_NTH == 0);
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
  f32x4 acc[PARTS][NT];
#pragma unroll
  for (int q = 0; q < PARTS; q++)
#pragma unroll
    for (int t = 0; t < NT; t++) acc[q][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  unsigned mypairs = 0;
  const int4* __restrict__ otab = orbtab + cls * NORB;
  uint32_t src[4];    // boxes of the product about to run, in 64-byte units
  f32x4 hand[4][2];   // this lane's words of its first step
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
  // the sources found for the next product, and its first step's words
  auto take = [&](const int (&id)[4], int cnt) __attribute__((always_inline)) {
    bool a = false;
    auto one = [&](int s) __attribute__((always_inline)) {
      a = a || id[s] >= 0;
      if (id[s] >= 0 && (l & 3) == 0) mypairs++;
      return (uint32_t)(id[s] >= 0 ? id[s] : nbj) * (uint32_t)(G::BS / 16);
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
  // a step's fragments into LDS buffer b; sync() waits for them
  auto copy = [&](const u32x4* from, int b) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < CH; e += GEN_NTH) lds_copy16(as_base + (b * CH + e + w * 64) * 16, from + e + tid);
  };
  auto op_src = [&](int o) __attribute__((always_inline)) -> const u32x4* { return opH + (size_t)(otab[o].w & 0xff) * FRO; };
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
    copy(op_src(o), 0);
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
    f32x4 ld[NS][2];
    uint32_t box[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) box[s] = src[s], ld[s][0] = hand[s][0], ld[s][1] = hand[s][1];
    auto next_product = [&]() __attribute__((always_inline)) {
      if (more) take(id, cntn);
      else any = false;
      first(cntn);
    };
    auto turned = [&](float(&raw)[NS][4], int h) __attribute__((always_inline)) {
      if constexpr (NS == 1) {
        f32x4 u = ld[0][h];
        asm volatile("ds_write_b128 %1, %0\n\tds_read_b128 %0, %2\n\ts_waitcnt lgkmcnt(0)"
                     : "+v"(u)
                     : "v"(turn_w), "v"(turn_r)
                     : "memory");
#pragma unroll
        for (int t = 0; t < 4; t++) raw[0][t] = u[t];
      } else {
#pragma unroll
        for (int q = 0; q < NS; q += 2) {
          f32x4 u = ld[q][h], v = ld[q + 1][h];
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
    // step s; XT: the last octet of the larger classes; LAST: the product's last step
    auto step = [&](int s, auto xt, auto lc) __attribute__((always_inline)) {
      constexpr bool XT = decltype(xt)::value, LAST = decltype(lc)::value;
      constexpr int qc0 = L.qc[0], qc1 = L.qc[1], qc2 = L.qc[2], qc3 = L.qc[3];
      constexpr int kc[8] = {XT ? qc0 : 0, XT ? qc1 : 1, XT ? qc2 : 2, XT ? qc3 : 3,
                             XT ? qc0 : 4, XT ? qc1 : 5, XT ? qc2 : 6, XT ? qc3 : 7};
      copy(LAST ? anext : acur + (size_t)(s + 1) * CH, buf ^ 1);
      if (!run) {
        if constexpr (LAST) next_product();
        return;
      }
      const u32x4* Ab = As + buf * CH + l;
#pragma unroll
      for (int part = 0; part < PARTS; part++) {
        u32x4 bh[NS], bl[NS];
#pragma unroll
        for (int h = 0; h < 2; h++) {
          float raw[NS][4];
          turned(raw, h);
#pragma unroll
          for (int t = 0; t < 4; t++) wht<J>(raw, t);
#pragma unroll
          for (int c = 0; c < NS; c++)
#pragma unroll
            for (int a = 2 * h; a < 2 * h + 2; a++) {
              const float e0 = raw[c ^ sub_rank(D, kc[2 * a] & D)][2 * a - 4 * h];
              const float e1 = raw[c ^ sub_rank(D, kc[2 * a + 1] & D)][2 * a + 1 - 4 * h];
              bh[c][a] = hi_pair(e0, e1);
              bl[c][a] = lo_pair(e0, e1, bh[c][a]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // the words of the next part, step or product
        if (part + 1 < PARTS || !LAST) {
          const int u = part + 1 < PARTS ? (part + 1) * 2 * NSTEP + 2 * s : 2 * (s + 1);
#pragma unroll
          for (int q = 0; q < NS; q++) ld[q][0] = unit(box[q], u), ld[q][1] = unit(box[q], u + 1);
        } else {
          next_product();
        }
        __builtin_amdgcn_sched_barrier(0);
        // a tile's fragments are read while the products of the one before run
        h8 fn[2][PARTS][2];
        auto fetch = [&](int t) __attribute__((always_inline)) {
#pragma unroll
          for (int q = 0; q < 2 * PARTS; q++)
            fn[t & 1][q / 2][q % 2] = __builtin_bit_cast(h8, Ab[(t * PARTS * 2 + q) * 64]);
        };
        fetch(0);
#pragma unroll
        for (int t = 0; t < NT; t++) {
          __builtin_amdgcn_sched_barrier(0);
          if (t + 1 < NT) fetch(t + 1);
          __builtin_amdgcn_sched_barrier(0);
          const h8 fh[2] = {fn[t & 1][0][0], fn[t & 1][PARTS - 1][0]}, fl[2] = {fn[t & 1][0][1], fn[t & 1][PARTS - 1][1]};
          const int c = sub_rank(D, L.tcls[t] & D);
          const u32x4 vh = bh[c], vl = bl[c];
          const h8 hi = __builtin_bit_cast(h8, vh), lo = __builtin_bit_cast(h8, vl);
          acc[part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[0], hi, acc[part][t], 0, 0, 0);
          // Im += S R; Re -= S I: the operand's sign bits
          const uint32_t sg = part ? 0x80008000u : 0u;
          const h8 hs = part ? __builtin_bit_cast(h8, vh ^ sg) : hi, ls = part ? __builtin_bit_cast(h8, vl ^ sg) : lo;
          acc[1 - part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[1], hs, acc[1 - part][t], 0, 0, 0);
          acc[part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fl[0], hi, acc[part][t], 0, 0, 0);
          acc[1 - part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fl[1], hs, acc[1 - part][t], 0, 0, 0);
          acc[part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[0], lo, acc[part][t], 0, 0, 0);
          acc[1 - part][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fh[1], ls, acc[1 - part][t], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
#pragma unroll 1
    for (int s = 0; s < NSTEP - 1; s++) {
      step(s, std::false_type{}, std::false_type{});
      sync();
      buf ^= 1;
    }
    step(NSTEP - 1, std::integral_constant<bool, G::XTRA != 0>{}, std::true_type{});
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

  if (tord >= 0) {
    const int oexp = -(orbit_exp(Q.mmax + (gsh >= 0 ? Q.ikey[tord] >> (3 * gsh) : 0u)) + Q.sa_e);
    f32x4* dst = reinterpret_cast<f32x4*>(Q.part + ((size_t)split * nb + tord) * G::ROWS + 4 * kq);
#pragma unroll
    for (int q = 0; q < PARTS; q++)
#pragma unroll
      for (int t = 0; t < NT; t++)
        dst[4 * (q * NT + t)] = f32x4{ldexpf(acc[q][t][0], oexp), ldexpf(acc[q][t][1], oexp), ldexpf(acc[q][t][2], oexp),
                                      ldexpf(acc[q][t][3], oexp)};
  }
  if (mypairs) atomicAdd(Q.npairs, (unsigned long long)mypairs);
}

// the partial sums of every level into the locals, splits in fixed order
struct GReduce {
  const float* part[MAXL + 1];
  float* L[MAXL + 1];
  unsigned off[MAXL + 2];
  int nsplit[MAXL + 1], nb[MAXL + 1], init[MAXL + 1];
  int nl;
};
template <int P>
__global__ __launch_bounds__(256) void k_gen_reduce(GReduce R) {
  using G = GConst<P>;
  constexpr int N = G::PARTS * G::P2;
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  const unsigned b = (unsigned)(t / N);
  const int i = (int)(t % N);
  if (t >= (size_t)R.off[R.nl] * N) return;
  int k = 0;
  while (k + 1 < R.nl && b >= R.off[k + 1]) k++;
  const unsigned bl = b - R.off[k];
  const float* p = R.part[k] + (size_t)bl * G::ROWS + c_gtab<P>.pos[i];
  float* L = R.L[k] + (size_t)bl * N + i;
  float s = R.init[k] ? 0.f : *L;
  for (int q = 0; q < R.nsplit[k]; q++) s += p[(size_t)q * R.nb[k] * G::ROWS];
  *L = s;
}

template <typename F>
int dispatch_gen(int p, F&& f) {
  switch (p) {
#define FMMX_CASE(P) \
  case P:            \
    return f(std::integral_constant<int, P>{});
    FMMX_CASE(4) FMMX_CASE(6) FMMX_CASE(8) FMMX_CASE(10) FMMX_CASE(12)
#undef FMMX_CASE
  }
  return fail(FMMX_EUNSUPPORTED, "order without an orbit M2L");
}

}  // namespace

int launch_orbit_gen_order(int p, const MSplitLevels& S, hipStream_t stream) {
  return dispatch_gen(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    using G = GConst<P>;
    const long n = S.off[S.nl] * G::BS, n8 = S.off[S.nl] * (G::PARTS * MLayout<P>::VS / 8);
    k_gzero<<<(S.nl * S.ng + 255) / 256, 256, 0, stream>>>(S);
    k_gmax<P><<<(int)((n8 + 255) / 256), 256, 0, stream>>>(S);
    k_gorder<P><<<(int)((n + 255) / 256), 256, 0, stream>>>(S);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "orbit M2L reorder launch failed");
  });
}

int launch_m2l_orbit_gen(int p, const M2LLaunch& A, int nwg, const int4* orbtab, hipStream_t stream) {
  return dispatch_gen(p, [&](auto pc) -> int {
    k_m2l_og<decltype(pc)::value><<<nwg, GEN_NTH, 0, stream>>>(A, orbtab);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "orbit M2L launch failed");
  });
}

int launch_orbit_gen_reduce(int p, const M2LLaunch& A, hipStream_t stream) {
  return dispatch_gen(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    GReduce R{};
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
    const long n = (long)R.off[R.nl] * GConst<P>::PARTS * P * P;
    k_gen_reduce<P><<<(int)((n + 255) / 256), 256, 0, stream>>>(R);
    return hipGetLastError() == hipSuccess ? FMMX_OK : fail(FMMX_EDEVICE, "orbit M2L reduction launch failed");
  });
}

}  // namespace fmmx
