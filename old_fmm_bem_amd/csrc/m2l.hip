// m2l.hip -- M2L (kernel/m2l.cxx) for CDNA4 (gfx950): targets of one parity
// class share the same 189 lattice offsets, so a tile of targets runs as 189
// GEMMs (operator [p^2 x p^2] x gathered source multipoles [p^2 x tile]); FP32
// on MFMA, every level in one launch.  The launchers of the FP16 and
// orbit forms (m2l_split.hip, m2l_orbit.hip, m2l_orbit_gen.hip,
// m2l_orbit_fp64.hip) are here too.
#include "phases.h"

namespace fmmx {

namespace {

// ---------------------------------------------------------------------
// M2L on MFMA.  A workgroup (WPG waves) owns a tile of 16 WPG targets of one
// parity class at a level; all of them see the same 189 lattice offsets
// (fmm/ijbox.cxx:366-401).  Per offset the operator (p^2 x p^2, stored by the
// host in MFMA fragment order) is staged once in LDS and each wave runs
// ceil(p^2/16) x ceil(p^2/4) v_mfma 16x16x4 steps for its 16 targets, the
// source multipoles (gathered through the dense key->box table) feeding the
// B operand straight from registers.  With nsplit > 1 the offsets are split
// over workgroups and the partial sums reduced by k_m2l_reduce in fixed
// order (deterministic).
constexpr int M2L_TN = 64;  // targets per workgroup of the FP64 vector kernel

// FP32 MFMA kernel: NT N-tiles (16 targets each) per wave, 4 waves, so a
// workgroup owns 64*NT targets.  With PA the next offset's operator
// fragments are prefetched into registers while the current offset runs on
// the matrix cores; the next offset's source multipoles always are
// (software pipelining).  The operator goes through one LDS buffer shared by
// the 4 waves.
template <int P, int NT, int PA, int WPG>
__global__ __launch_bounds__(64 * WPG) void k_m2l(M2LLaunch A) {
  // this workgroup's level (uniform selects: no dynamic indexing of the
  // kernel arguments)
  M2LLev Q = A.lv[0];
#pragma unroll
  for (int k = 1; k < MAXL + 1; k++)
    if (k < A.nlv && (int)blockIdx.x >= A.lv[k].wg0) Q = A.lv[k];
  const int lev = Q.lev, nb = Q.nb, nsplit = Q.nsplit, init = Q.init, region = Q.region, gsh = Q.gsh;
  const int* __restrict__ cls_cnt = Q.cls_cnt;
  const uint32_t* __restrict__ ord = Q.ord;
  const uint32_t* __restrict__ ikey = Q.ikey;
  const int* __restrict__ dense_j = Q.dense_j;
  const float* __restrict__ M = Q.M;
  float* __restrict__ L = Q.L;
  float* __restrict__ part = Q.part;
  const float* __restrict__ opF = Q.opF;
  const int4* __restrict__ offtab = Q.offtab;
  unsigned long long* __restrict__ npairs = Q.npairs;
  const int bid = (int)blockIdx.x - Q.wg0, nwg = Q.nwg;
  using T = float;
  using ML = MLayout<P>;
  constexpr int P2 = P * P, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, FR = KS * MT * 64;
  constexpr int NTH = 64 * WPG;          // threads per workgroup
  constexpr int TN = 16 * NT * WPG;      // targets per workgroup
  constexpr int NV = FR / 4;             // float4 per operator
  constexpr int NVT = (NV + NTH - 1) / NTH;  // float4 per thread
  using V4 = f32x4;
  // PA 2: two operator buffers (the next offset's operator is written to one
  // while the MFMAs read the other; one barrier per offset)
  constexpr int NBUF = PA == 2 ? 2 : 1;
  __shared__ __align__(16) T As[NBUF * FR];
  __shared__ int s_class, s_start, s_n;
  const int tid = threadIdx.x;
  // XCD-aware order: workgroups are dispatched round-robin over the 8 XCDs,
  // so workgroup b runs on XCD b%8; class b%8 keeps each XCD's L2 on one
  // parity class's 189 operators.  Work item k = b/8 of that class, split
  // major: the workgroups resident on an XCD at a time share one split's
  // 189/nsplit operators, which then stay in its L2 across tiles.
  // With region set, workgroup b runs on XCD b%8 for a block of tiles
  // instead: XCD x owns tiles [x*tpr, (x+1)*tpr) of every class, so the 8
  // siblings of a box (one per class) run on one XCD and share their source
  // multipoles in its L2; items on an XCD go tile-major, then split, then
  // class.
  int cls0, split, tile;
  // (level ranges start at multiples of 8, so bid % 8 is still the XCD)
  if (region) {
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
    for (int c = 0; c < cls0; c++) start += cls_cnt[c];
    const int cnt = cls_cnt[cls0], nt = (cnt + TN - 1) / TN;
    s_class = tile < nt ? cls0 : -1;
    s_start = start + tile * TN;
    s_n = tile < nt ? min(TN, cnt - tile * TN) : 0;
  }
  __syncthreads();
  const int cls = s_class, ntile = s_n;
  if (cls < 0) return;
  const int w = tid >> 6, l = tid & 63, j = l & 15, kq = l >> 4;
  const int g = 1 << lev;
  int tord[NT], tx[NT], ty[NT], tz[NT];
#pragma unroll
  for (int n = 0; n < NT; n++) {
    const int t = (w * NT + n) * 16 + j;
    tord[n] = -1;
    tx[n] = ty[n] = tz[n] = 0;
    if (t < ntile) {
      tord[n] = (int)ord[s_start + t];
      morton_decode(ikey[tord[n]], lev, tx[n], ty[n], tz[n]);
    }
  }
  const bool wave_on = w * NT * 16 < ntile;
  const int per = (NEBM + nsplit - 1) / nsplit, o0 = split * per, o1 = min(NEBM, o0 + per);
  V4 acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; n++)
#pragma unroll
    for (int mt = 0; mt < MT; mt++) acc[n][mt] = V4{0.f, 0.f, 0.f, 0.f};
  unsigned long long mypairs = 0;
  float4 areg[PA ? NVT : 1];  // PA 1: unsigned operator prefetch; PA 2: signed
  // Reflected offsets use the operator of the canonical offset with element
  // (row i, col k) times T_r(i) T_r(k).  The float4s a thread stages sit at
  // fixed places, so their sign patterns are worked out once: nibble r of
  // sgn[v] flags the 4 floats of the thread's v-th float4 under reflection r.
  // Fragment element q = (ks * MT + mt) * 64 + lane holds row 16 mt + lane % 16
  // and col (lane / 16) * KS + ks.
  uint32_t sgn[PA == 1 ? 1 : NVT];
  if (PA != 1) {
    constexpr ReflMask<P> RM{};
#pragma unroll
    for (int v = 0; v < NVT; v++) {
      sgn[v] = 0;
      const int e = tid + NTH * v;
      if (e < NV) {
        const int q = 4 * e, lane = q & 63, mt = (q >> 6) % MT, ks = (q >> 6) / MT;
        const int col = (lane >> 4) * KS + ks, row0 = 16 * mt + (lane & 15);
        for (int r = 1; r < 8; r++) {
          const bool cn = col < P2 && RM.neg(r, col);
          for (int jj = 0; jj < 4; jj++)
            if (row0 + jj < P2 && RM.neg(r, row0 + jj) != cn) sgn[v] |= 1u << (4 * r + jj);
        }
      }
    }
  }
  T bcur[NT][KS];
#define FMMX_LOAD_B(o_, dst_)                                                                 \
  {                                                                                           \
    const int4 off_ = offtab[cls * NEBM + (o_)];                                              \
    _Pragma("unroll") for (int n = 0; n < NT; n++) {                                          \
      int s_ = -1;                                                                            \
      if (tord[n] >= 0) {                                                                     \
        const int jx = tx[n] - off_.x, jy = ty[n] - off_.y, jz = tz[n] - off_.z;              \
        if (jx >= 0 && jx < g && jy >= 0 && jy < g && jz >= 0 && jz < g &&                    \
            (gsh < 0 || !((jx ^ tx[n]) >> gsh | (jy ^ ty[n]) >> gsh | (jz ^ tz[n]) >> gsh)))   \
          s_ = dense_j[morton_encode(jx, jy, jz, lev)];                                       \
      }                                                                                       \
      if (s_ >= 0 && kq == 0) mypairs++;                                                      \
      any_ = any_ || s_ >= 0;                                                                 \
      const float4* ms_ = reinterpret_cast<const float4*>(M + (size_t)(s_ >= 0 ? s_ : 0) * ML::VS + kq * ML::KSP); \
      _Pragma("unroll") for (int v4 = 0; v4 < ML::KSP / 4; v4++) {                            \
        const float4 m4 = s_ >= 0 ? ms_[v4] : make_float4(0.f, 0.f, 0.f, 0.f);                \
        if (4 * v4 + 0 < KS) dst_[n][4 * v4 + 0] = (kq * KS + 4 * v4 + 0 < P2) ? m4.x : 0.f;  \
        if (4 * v4 + 1 < KS) dst_[n][4 * v4 + 1] = (kq * KS + 4 * v4 + 1 < P2) ? m4.y : 0.f;  \
        if (4 * v4 + 2 < KS) dst_[n][4 * v4 + 2] = (kq * KS + 4 * v4 + 2 < P2) ? m4.z : 0.f;  \
        if (4 * v4 + 3 < KS) dst_[n][4 * v4 + 3] = (kq * KS + 4 * v4 + 3 < P2) ? m4.w : 0.f;  \
      }                                                                                       \
    }                                                                                         \
  }
#define FMMX_LOAD_A(o_)                                                                       \
  {                                                                                           \
    const float4* src_ = reinterpret_cast<const float4*>(opF + (size_t)(offtab[cls * NEBM + (o_)].w & 0xffff) * FR); \
    _Pragma("unroll") for (int v = 0; v < NVT; v++) {                                         \
      const int e = tid + NTH * v;                                                            \
      if (e < NV) areg[v] = src_[e];                                                          \
    }                                                                                         \
  }
#define FMMX_LOAD_AS(o_)                                                                      \
  {                                                                                           \
    const int w_ = offtab[cls * NEBM + (o_)].w, r_ = w_ >> 16;                                \
    const float4* src_ = reinterpret_cast<const float4*>(opF + (size_t)(w_ & 0xffff) * FR);   \
    _Pragma("unroll") for (int v = 0; v < NVT; v++) {                                         \
      const int e = tid + NTH * v;                                                            \
      if (e < NV) {                                                                           \
        float4 x_ = src_[e];                                                                  \
        const uint32_t nib_ = sgn[v] >> (4 * r_);                                             \
        x_.x = __uint_as_float(__float_as_uint(x_.x) ^ ((nib_ & 1u) << 31));                  \
        x_.y = __uint_as_float(__float_as_uint(x_.y) ^ (((nib_ >> 1) & 1u) << 31));           \
        x_.z = __uint_as_float(__float_as_uint(x_.z) ^ (((nib_ >> 2) & 1u) << 31));           \
        x_.w = __uint_as_float(__float_as_uint(x_.w) ^ (((nib_ >> 3) & 1u) << 31));           \
        areg[v] = x_;                                                                         \
      }                                                                                       \
    }                                                                                         \
  }
#define FMMX_STORE_A(buf_)                                                                    \
  {                                                                                           \
    _Pragma("unroll") for (int v = 0; v < NVT; v++) {                                         \
      const int e = tid + NTH * v;                                                            \
      if (e < NV) reinterpret_cast<float4*>(As + (buf_) * FR)[e] = areg[v];                   \
    }                                                                                         \
  }
  if constexpr (PA == 2) {
    // double-buffered operator: load offset o+1's operator (signed) and
    // source multipoles into registers, run offset o's MFMAs from one LDS
    // buffer, write o+1's operator into the other, one barrier
    bool cur_any = false;
    if (o0 < o1) {
      FMMX_LOAD_AS(o0);
      FMMX_STORE_A(0);
      bool any_ = false;
      FMMX_LOAD_B(o0, bcur);
      cur_any = __ballot(any_) != 0;
    }
    __syncthreads();
    int buf = 0;
    for (int o = o0; o < o1; o++) {
      T bnext[NT][KS];
      bool next_any = false;
      if (o + 1 < o1) {
        FMMX_LOAD_AS(o + 1);
        bool any_ = false;
        FMMX_LOAD_B(o + 1, bnext);
        next_any = __ballot(any_) != 0;
      }
      if (wave_on && cur_any) {
        const T* Ab = As + buf * FR;
      T af[2][MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) af[0][mt] = Ab[mt * 64 + l];
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        if (ks + 1 < KS) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) af[(ks + 1) & 1][mt] = Ab[((ks + 1) * MT + mt) * 64 + l];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int n = 0; n < NT; n++) acc[n][mt] = Mfma<T>::fma(af[ks & 1][mt], bcur[n][ks], acc[n][mt]);
        __builtin_amdgcn_sched_barrier(0);
      }
      }
      if (o + 1 < o1) FMMX_STORE_A(buf ^ 1);
      __syncthreads();
      if (o + 1 < o1) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
          for (int ks = 0; ks < KS; ks++) bcur[n][ks] = bnext[n][ks];
        cur_any = next_any;
      }
      buf ^= 1;
    }
  } else {
  // a wave skips the MFMAs of an offset for which none of its 16 targets has
  // a source box (boundary tiles); the vote keeps the branch wave-uniform
  bool cur_any = false;
  if (o0 < o1) {
    if (PA) FMMX_LOAD_A(o0);
    bool any_ = false;
    FMMX_LOAD_B(o0, bcur);
    cur_any = __ballot(any_) != 0;
  }
  for (int o = o0; o < o1; o++) {
    __syncthreads();  // every wave is done with the previous operator
    if (PA) {
#pragma unroll
      for (int v = 0; v < NVT; v++) {
        const int e = tid + NTH * v;
        if (e < NV) reinterpret_cast<float4*>(As)[e] = areg[v];
      }
    } else {
      const int w = offtab[cls * NEBM + o].w, refl = w >> 16;
      const float4* src = reinterpret_cast<const float4*>(opF + (size_t)(w & 0xffff) * FR);
#pragma unroll
      for (int v = 0; v < NVT; v++) {
        const int e = tid + NTH * v;
        if (e < NV) {
          float4 x = src[e];
          const uint32_t nib = sgn[v] >> (4 * refl);
          x.x = __uint_as_float(__float_as_uint(x.x) ^ ((nib & 1u) << 31));
          x.y = __uint_as_float(__float_as_uint(x.y) ^ (((nib >> 1) & 1u) << 31));
          x.z = __uint_as_float(__float_as_uint(x.z) ^ (((nib >> 2) & 1u) << 31));
          x.w = __uint_as_float(__float_as_uint(x.w) ^ (((nib >> 3) & 1u) << 31));
          reinterpret_cast<float4*>(As)[e] = x;
        }
      }
    }
    __syncthreads();
    T bnext[NT][KS];
    bool next_any = false;
    if (o + 1 < o1) {
      if (PA) FMMX_LOAD_A(o + 1);
      bool any_ = false;
      FMMX_LOAD_B(o + 1, bnext);
      next_any = __ballot(any_) != 0;
    }
    if (wave_on && cur_any) {
      // operator fragments of step ks+1 are read from LDS while the MFMAs of
      // step ks run; the scheduling barriers keep that order, so the LDS
      // latency sits behind MT matrix instructions instead of in front of one
      const T* Ab = As;
      T af[2][MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) af[0][mt] = Ab[mt * 64 + l];
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        if (ks + 1 < KS) {
#pragma unroll
          for (int mt = 0; mt < MT; mt++) af[(ks + 1) & 1][mt] = Ab[((ks + 1) * MT + mt) * 64 + l];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int n = 0; n < NT; n++) acc[n][mt] = Mfma<T>::fma(af[ks & 1][mt], bcur[n][ks], acc[n][mt]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (o + 1 < o1) {
#pragma unroll
      for (int n = 0; n < NT; n++)
#pragma unroll
        for (int ks = 0; ks < KS; ks++) bcur[n][ks] = bnext[n][ks];
      cur_any = next_any;
    }
  }
  }
#undef FMMX_LOAD_AS
#undef FMMX_STORE_A
#undef FMMX_LOAD_A
#undef FMMX_LOAD_B
#pragma unroll
  for (int n = 0; n < NT; n++) {
    if (tord[n] < 0) continue;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 16 * mt + 4 * kq + r;
        if (i < P2) {
          const T v = acc[n][mt][r];
          if (nsplit == 1) {
            T* dst = L + (size_t)tord[n] * P2 + i;
            *dst = init ? v : *dst + v;
          } else {
            part[((size_t)split * nb + tord[n]) * P2 + i] = v;
          }
        }
      }
  }
  if (mypairs) atomicAdd(npairs, mypairs);
}

// FP64 M2L on the vector FMA units, for what the orbit form (m2l_orbit_fp64.hip)
// is not built for: the REF convention, orders below 6 and 18, the Yukawa and
// Helmholtz kernels.  Same tiles and offset split as k_m2l; per offset the operator
// (k-major) and the gathered source multipoles go through LDS in K-chunks
// and each thread accumulates a (rows x 4 targets) register block.
constexpr int M2LV_KC = 32, M2LV_BST = M2L_TN + 4;

// PARTS 2 (Helmholtz): split expansions, D = 2 p^2 rows and k-indices; the
// multipole part t of box s sits at s * 2 VS + t * VS in the padded layout.
template <int P, typename T, int PARTS = 1>
__global__ __launch_bounds__(256) void k_m2l_vec(int lev, int nb, int nsplit, const int* __restrict__ cls_cnt,
                                                 const uint32_t* __restrict__ ord, const uint32_t* __restrict__ ikey,
                                                 const int* __restrict__ dense_j, const T* __restrict__ M,
                                                 T* __restrict__ L, T* __restrict__ part, const T* __restrict__ opT,
                                                 const int4* __restrict__ offtab, int init, int gsh,
                                                 unsigned long long* __restrict__ npairs) {
  using ML = MLayout<P>;
  constexpr int P2 = P * P, D = PARTS * P2, RPT = (D + 15) / 16;
  constexpr int KC = D * (int)sizeof(T) > 1200 ? M2LV_KC / 2 : M2LV_KC;  // LDS within 64 KB
  __shared__ T As[KC][D];
  __shared__ T Bs[KC][M2LV_BST];
  __shared__ int tpos[M2L_TN][3];
  __shared__ int tord[M2L_TN];
  __shared__ int src[M2L_TN];
  __shared__ int s_class, s_start, s_n;
  const int tid = threadIdx.x;
  const int tile = blockIdx.x / nsplit, split = blockIdx.x % nsplit;
  if (tid == 0) {
    int w = tile, start = 0, cls = -1, n = 0;
    for (int c = 0; c < 8; c++) {
      const int cnt = cls_cnt[c], nt = (cnt + M2L_TN - 1) / M2L_TN;
      if (cls < 0 && w < nt) {
        cls = c;
        n = min(M2L_TN, cnt - w * M2L_TN);
        start += w * M2L_TN;
      } else if (cls < 0) {
        w -= nt;
        start += cnt;
      }
    }
    s_class = cls;
    s_start = start;
    s_n = n;
  }
  __syncthreads();
  const int cls = s_class, ntile = s_n;
  if (cls < 0) return;
  const int g = 1 << lev;
  if (tid < M2L_TN) {
    int ix = -1000, iy = -1000, iz = -1000, o = -1;
    if (tid < ntile) {
      o = (int)ord[s_start + tid];
      morton_decode(ikey[o], lev, ix, iy, iz);
    }
    tpos[tid][0] = ix;
    tpos[tid][1] = iy;
    tpos[tid][2] = iz;
    tord[tid] = o;
  }
  const int tx = tid & 15, ty = tid >> 4;
  T acc[RPT][4];
#pragma unroll
  for (int r = 0; r < RPT; r++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[r][c] = T(0);
  unsigned long long mypairs = 0;
  const int per = (NEBM + nsplit - 1) / nsplit, o0 = split * per, o1 = min(NEBM, o0 + per);
  for (int oi = o0; oi < o1; oi++) {
    const int4 off = offtab[cls * NEBM + oi];
    __syncthreads();
    int has = 0;
    if (tid < M2L_TN) {
      int s = -1;
      if (tid < ntile) {
        const int ix = tpos[tid][0], iy = tpos[tid][1], iz = tpos[tid][2];
        const int jx = ix - off.x, jy = iy - off.y, jz = iz - off.z;
        if (jx >= 0 && jx < g && jy >= 0 && jy < g && jz >= 0 && jz < g &&
            (gsh < 0 || !((jx ^ ix) >> gsh | (jy ^ iy) >> gsh | (jz ^ iz) >> gsh)))
          s = dense_j[morton_encode(jx, jy, jz, lev)];
      }
      src[tid] = s;
      has = s >= 0;
      if (s >= 0) mypairs++;
    }
    // no target of the tile has a source box at this offset (domain edge,
    // sparse surfaces): neither stage the operator nor multiply
    if (!__syncthreads_or(has)) continue;
    const T* A = opT + (size_t)off.w * D * D;
    for (int k0 = 0; k0 < D; k0 += KC) {
      const int kc = min(KC, D - k0);
      __syncthreads();
      for (int e = tid; e < kc * D; e += 256) As[e / D][e % D] = A[(size_t)k0 * D + e];
      for (int e = tid; e < kc * M2L_TN; e += 256) {
        const int t = e / kc, k = k0 + e % kc, s = src[t];
        const int part = PARTS == 1 ? 0 : k / P2, kk = PARTS == 1 ? k : k % P2;
        Bs[e % kc][t] = s >= 0 ? M[(size_t)s * PARTS * ML::VS + part * ML::VS + ML::at(kk)] : T(0);
      }
      __syncthreads();
      for (int k = 0; k < kc; k++) {
        T bv[4];
#pragma unroll
        for (int c = 0; c < 4; c++) bv[c] = Bs[k][tx * 4 + c];
#pragma unroll
        for (int r = 0; r < RPT; r++) {
          const int row = ty + 16 * r;
          const T av = row < D ? As[k][row] : T(0);
#pragma unroll
          for (int c = 0; c < 4; c++) acc[r][c] += av * bv[c];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int t = tx * 4 + c;
    if (t >= ntile) continue;
#pragma unroll
    for (int r = 0; r < RPT; r++) {
      const int row = ty + 16 * r;
      if (row >= D) continue;
      if (nsplit == 1) {
        T* dst = L + (size_t)tord[t] * D + row;
        *dst = init ? acc[r][c] : *dst + acc[r][c];
      } else {
        part[((size_t)split * nb + tord[t]) * D + row] = acc[r][c];
      }
    }
  }
  if (tid < M2L_TN && mypairs) atomicAdd(npairs, mypairs);
}

// the reductions of several levels in one launch: elements [off[k], off[k+1])
// belong to level k (same order of the split sums as k_m2l_reduce, init 1)
struct ReduceLevels {
  const float* part[MAXL + 1];
  float* L[MAXL + 1];
  long off[MAXL + 2];
  int nsplit[MAXL + 1];
  int nl;
};
__global__ void k_m2l_reduce_levels(ReduceLevels R) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= R.off[R.nl]) return;
  int k = 0;
  while (k + 1 < R.nl && t >= R.off[k + 1]) k++;
  const long n = R.off[k + 1] - R.off[k], e = t - R.off[k];
  const float* part = R.part[k];
  float s = 0.f;
  for (int j = 0; j < R.nsplit[k]; j++) s += part[(size_t)j * n + e];
  R.L[k][e] = s;
}

template <typename T>
__global__ void k_zero_t(long n, T* __restrict__ a) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = T(0);
}

}  // namespace

// Offset splits of the M2L launch at a level (partial sums when > 1).
Engine::M2LVariant Engine::m2l_variant(int lev) const {
  M2LVariant v = tune[lev];
  if (lev != lmax && m2l_all_levels()) {
    // one launch for all levels: the leaf level's shape, this level's splits
    const M2LVariant lf = m2l_variant(lmax);
    v.nt = lf.nt;
    v.pa = lf.pa;
    v.wpg = lf.wpg;
  }
  if (v.nt <= 0) v.nt = 1;
  // default: the FP16 split kernel where it applies (FP32 Laplace engine,
  // EXACT, p 6..12), else LDS staging
  if (v.pa < 0) v.pa = (split_ok && !yk && !hh && !fp64) ? (orb_ok && orbit_fits() ? 6 : wide_ok ? 5 : 4) : 0;
  if (v.wpg <= 0) v.wpg = 8;
  if (const char* e = getenv("FMMX_M2L_NT")) v.nt = atoi(e) == 4 ? 4 : atoi(e) == 2 ? 2 : 1;
  if (const char* e = getenv("FMMX_M2L_PA")) v.pa = std::max(0, std::min(6, atoi(e)));
  if (const char* e = getenv("FMMX_M2L_WPG")) v.wpg = atoi(e) == 4 ? 4 : atoi(e) == 16 ? 16 : 8;
  if (v.pa >= 3) {
    // FP16 split kernel: Laplace FP32 engine, p 6..12; two operator buffers
    // with one N-tile and 8 waves where they fit LDS
    if (!split_ok || yk || hh || fp64) v.pa = 0;
    else if (v.pa == 6 && !(orb_ok && orbit_fits())) v.pa = wide_ok ? 5 : 4;
    else if (v.pa == 5 && !wide_ok) v.pa = 4;
    if (v.pa == 6) v.nt = 1, v.wpg = ORB_WPG;
    if (v.pa == 4 && !split_db_fits(p)) v.pa = 3;
    // 32 targets per wave: 8 waves (two buffers) or 4 (one); 64 targets per
    // wave (nt 4): 4 waves, two buffers
    if (v.pa == 5) {
      if (v.nt == 4) v.wpg = 4;
      else v.nt = 2, v.wpg = v.wpg == 4 ? 4 : 8;
    }
    if (v.pa != 5 && v.nt == 4) v.nt = 2;
    if (v.pa == 4) v.wpg = v.nt == 2 ? 4 : 8;  // 8 waves of one N-tile or 4 of two
    if (v.pa == 3 && v.nt == 2) v.wpg = 4;
    if (v.wpg == 16) v.wpg = 8;
  }
  if (v.pa == 2 && (p > 11 || v.nt != 1)) v.pa = 0;  // two operator buffers fit LDS up to p = 11
  if (v.wpg == 16 && v.pa != 2) v.wpg = 8;
  // reflection-canonical operators are signed while staged: no register prefetch form
  if (v.pa == 1 && canon && !yk) v.pa = 0;
  if (v.pa < 3 && v.wpg == 16 && v.pa != 2) v.wpg = 8;
  if (const char* e = getenv("FMMX_M2L_SPLIT")) v.nsplit = atoi(e);
  if (const char* e = getenv("FMMX_M2L_SPLITS")) {
    // per level, comma-separated from level 2
    for (int l = 2; e && *e; l++) {
      if (l == lev) v.nsplit = atoi(e);
      e = strchr(e, ',');
      if (e) e++;
    }
  }
  if (v.nsplit <= 0) {
    // enough workgroups to cover the chip: split the 189 offsets when tiles are few
    if (fp64 && !orbit_f64()) {
      v.nsplit = 1024 / ((si.nb[lev] + M2L_TN - 1) / M2L_TN + 8);
    } else {
      int cmax = 0;
      for (int c = 0; c < 8; c++) cmax = std::max(cmax, cls_cnt_h[lev][c]);
      const int tpc = std::max(1, (cmax + 16 * v.wpg * v.nt - 1) / (16 * v.wpg * v.nt));
      v.nsplit = 1024 / (8 * tpc);
      // the orbit kernel: 63 products, and each workgroup starts with a copy
      // of most of an operator; levels of a few tiles gain from more than 8
      // splits (latency), larger ones lose (N = 1M, level 4 of 5: 8 splits
      // 0.331 ms for the launch, 16 splits 0.341; a sphere's leaf level of
      // 4,639 boxes 0.104 against 0.125)
      if (v.pa == 6 && tpc > 1) v.nsplit = std::min(v.nsplit, 8);
      // FP64 orbits: 512 workgroups of a level, each with its own share of the
      // 63 products (one workgroup per CU at a time)
      if (orbit_f64()) v.nsplit = 512 / (8 * tpc);
      // Helmholtz: one workgroup per CU and 1.5 KB of partial sums per target
      // and split (sphere of 1M points: 4 splits of the leaf level 1.68 ms for
      // M2L and L2L, 7 splits 1.84, 2 splits 1.85)
      if (hh) v.nsplit = std::max(1, std::min(640 / (8 * tpc), tpc > 1 ? 8 : 16));
    }
  }
  v.nsplit = std::max(1, std::min(16, v.nsplit));
  return v;
}

// MFMA M2L: the launch parameters of one level, its workgroups from wg0
// (grid = 8 classes x tiles x splits; a block of tiles per XCD once every XCD
// gets at least one tile)
M2LLev Engine::m2l_desc(int lev, int nt, int wpg, int nsplit, float* part, int init, int wg0) {
  M2LLev d{};
  const int MT = (P2 + 15) / 16, KS = (P2 + 3) / 4;
  const size_t FR = (size_t)KS * MT * 64;
  const size_t opoff = (yk || m2l_per_level) ? (size_t)(lev - 2) * NOFF * FR : 0;
  // reflection-canonical operators (Laplace, EXACT) are signed while staged
  const bool use_canon = canon && !yk;
  int cmax = 0;
  for (int c = 0; c < 8; c++) cmax = std::max(cmax, cls_cnt_h[lev][c]);
  const int tpc = std::max(1, (cmax + 16 * wpg * nt - 1) / (16 * wpg * nt));
  int region = tpc >= 8 ? 1 : 0;
  if (const char* e = getenv("FMMX_M2L_REGION")) region = region && atoi(e) != 0;
  d.cls_cnt = cls_cnt[lev].as<int>();
  d.ord = cls_ord[lev].as<uint32_t>();
  d.ikey = si.bkey[lev].as<uint32_t>();
  d.dense_j = sj.dense[lev].as<int>();
  d.M = mexp[lev].as<float>();
  d.L = lexp[lev].as<float>();
  d.part = part;
  d.opF = (yk ? yop_m2l : op_m2l).as<float>() + opoff;
  // FP16 split form: per-level operator sets in REF, one set otherwise
  const size_t frh = split_ok ? split_frag_count(p) : 0;
  d.Mh = mexp_h[lev].as<uint4>();
  d.opH = op_m2l_h.as<uint4>() + (m2l_per_level ? (size_t)(lev - 2) * NOFF * frh : 0);
  d.mmax = mmax_buf.as<unsigned>() + lev;
  d.sa_e = sa_e;
  d.offtab = (use_canon ? offtab_c : offtab).as<int4>();
  d.npairs = pair_ctr.as<unsigned long long>() + 2 + lev;
  d.lev = lev;
  d.nb = si.nb[lev];
  d.nbj = sj.nb[lev];
  d.nsplit = nsplit;
  d.init = init;
  d.region = region;
  d.gsh = group_shift(lev);
  d.wg0 = wg0;
  d.nwg = region ? 64 * ((tpc + 7) / 8) * nsplit : 8 * tpc * nsplit;
  return d;
}

// the k_m2l instance of a launch shape (N-tiles per wave, operator staging,
// waves per workgroup)
template <int P>
void launch_m2l(const M2LLaunch& A, int nwg, int nt, int pa, int wpg, hipStream_t stream) {
#define FMMX_M2L_LAUNCH(NT_, PA_, W_) k_m2l<P, NT_, PA_, W_><<<nwg, 64 * W_, 0, stream>>>(A)
  if (pa == 2 && P > 11) pa = 0;  // two operator buffers fit the 160 KB of LDS up to p = 11
  if (pa == 2) {
    if constexpr (P <= 11) {
      if (wpg == 16) FMMX_M2L_LAUNCH(1, 2, 16);
      else FMMX_M2L_LAUNCH(1, 2, 8);
    }
  } else if (wpg == 8) {
    if (nt == 1 && !pa) FMMX_M2L_LAUNCH(1, 0, 8);
    else if (nt == 1) FMMX_M2L_LAUNCH(1, 1, 8);
    else FMMX_M2L_LAUNCH(2, 0, 8);
  } else {
    if (nt == 1 && !pa) FMMX_M2L_LAUNCH(1, 0, 4);
    else if (nt == 1) FMMX_M2L_LAUNCH(1, 1, 4);
    else FMMX_M2L_LAUNCH(2, 0, 4);
  }
#undef FMMX_M2L_LAUNCH
}

// the orbit kernel addresses a level's stored boxes with 32-bit byte offsets
bool Engine::orbit_fits() const { return ((size_t)sj.nb[lmax] + 1) * orbit_box_floats(p) * 4 < ((size_t)1 << 32); }

bool Engine::m2l_split(int lev) const { return !fp64 && !hh && !yk && m2l_variant(lev).pa >= 3; }

// The FP16 split kernel's inputs for levels [l0, l1]: the multipoles of every
// level split into hi/lo pairs scaled by 2^(14 - exponent of the level's
// largest magnitude), one pair of launches for all levels
int Engine::run_msplit(int l0, int l1, int form) {
  MSplitLevels S{};
  S.off[0] = 0;
  S.wide = form == 6 ? 2 : form == 5 ? 1 : 0;
  int rc = mmax_buf.ensure((MAXL + 1) * 4);
  if (rc) return rc;
  for (int lev = l0; lev <= l1; lev++) {
    const int nb = sj.nb[lev];
    if (nb == 0 || si.nb[lev] == 0) continue;
    S.M[S.nl] = mexp[lev].as<float>();
    S.Mh[S.nl] = mexp_h[lev].as<uint4>();
    S.mmax[S.nl] = mmax_buf.as<unsigned>() + lev;
    S.off[S.nl + 1] = S.off[S.nl] + nb + 1;  // and the zero box
    S.nl++;
  }
  if (S.nl == 0) return FMMX_OK;
  return launch_msplit(p, S, stream);
}

// FP32 M2L of all levels l0..lmax in one launch, in the leaf level's launch
// shape with each level's offset splits: levels with splits write partial
// sums (reduced afterwards in fixed order), the others write their locals;
// the L2L chain then adds the parents' locals level by level.  With the FP16
// split shape (staging 3, 4) the multipoles are split first.
int Engine::run_m2l_all(int l0) {
  if (hh) return run_m2l_hh(l0, lmax, true);
  if (fp64) return run_m2l_f64(l0, lmax, true);
  const M2LVariant leaf = m2l_variant(lmax);
  const bool split = leaf.pa >= 3, orbit = leaf.pa == 6;
  // floats of a target's partial sums (the orbit form always goes through them)
  const size_t rows = orbit ? 8 * OLayout<2>::RW : P2;
  M2LLaunch A{};
  size_t need = 0;
  for (int lev = l0; lev <= lmax; lev++)
    if (si.nb[lev] > 0 && sj.nb[lev] > 0 && (orbit || m2l_splits(lev) > 1))
      need += (size_t)m2l_splits(lev) * si.nb[lev] * rows;
  int rc = m2l_part.ensure(std::max<size_t>(need, 1) * 4);
  if (rc) return rc;
  if (split && ((rc = upload_split(leaf.pa)) || (rc = run_msplit(l0, lmax, leaf.pa)))) return rc;
  size_t off = 0;
  int wg = 0;
  for (int lev = l0; lev <= lmax; lev++) {
    const int nb = si.nb[lev];
    if (nb == 0) continue;
    const long nl = (long)nb * P2;
    if (sj.nb[lev] == 0) {
      k_zero_t<float><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, lexp[lev].as<float>());
      continue;
    }
    const int ns = m2l_splits(lev);
    A.lv[A.nlv] = m2l_desc(lev, leaf.nt, leaf.wpg, ns, orbit || ns > 1 ? m2l_part.as<float>() + off : nullptr, 1, wg);
    if (orbit) A.lv[A.nlv].opH = op_m2l_o.as<uint4>();
    if (leaf.pa == 4) A.lv[A.nlv].offtab = offtab_s.as<int4>();
    if (leaf.pa == 5) {
      A.lv[A.nlv].offtab = offtab.as<int4>();
      A.lv[A.nlv].opH = op_m2l_w.as<uint4>();
    }
    wg += A.lv[A.nlv].nwg;
    A.nlv++;
    if (orbit || ns > 1) off += (size_t)ns * nb * rows;
  }
  if (A.nlv == 0) return FMMX_OK;
  return dispatch_p(p, [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    if (per_phase) FMMX_HIP(hipEventRecord(ev[8], stream));
    if (split) {
      int r2 = orbit          ? launch_m2l_orbit(p, A, wg, orbtab.as<int4>(), stream)
               : leaf.pa == 5 ? launch_m2l_wide(p, A, wg, leaf.wpg, leaf.nt, stream)
                              : launch_m2l_split(p, A, wg, leaf.nt, leaf.wpg, leaf.pa == 4, stream);
      if (r2) return r2;
    } else {
      launch_m2l<P>(A, wg, leaf.nt, leaf.pa, leaf.wpg, stream);
    }
    if (per_phase) {
      FMMX_HIP(hipEventRecord(ev[9], stream));
      m2l_timed = true;
    }
    if (orbit) return launch_orbit_reduce(p, A, stream);
    // the partial sums of every level with splits, one launch
    ReduceLevels R{};
    R.off[0] = 0;
    for (int k = 0; k < A.nlv; k++) {
      const M2LLev& d = A.lv[k];
      if (d.nsplit < 2) continue;
      R.part[R.nl] = d.part;
      R.L[R.nl] = d.L;
      R.nsplit[R.nl] = d.nsplit;
      R.off[R.nl + 1] = R.off[R.nl] + (long)d.nb * P2;
      R.nl++;
    }
    if (R.nl > 0)
      k_m2l_reduce_levels<<<(int)((R.off[R.nl] + 255) / 256), 256, 0, stream>>>(R);
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  });
}

// FP32 Helmholtz M2L of levels l0..l1 by reflection orbits, one launch; the
// locals are written (init) or added to
int Engine::run_m2l_hh(int l0, int l1, bool init) {
  M2LLaunch A{};
  MSplitLevels S{};
  const size_t rows = orbit_gen_rows(p), frg = orbit_gen_frags(p);
  size_t need = 0;
  for (int lev = l0; lev <= l1; lev++)
    if (si.nb[lev] > 0 && sj.nb[lev] > 0) need += (size_t)m2l_splits(lev) * si.nb[lev] * rows;
  int rc = m2l_part.ensure(std::max<size_t>(need, 1) * 4);
  // one scale per level and independent group
  const int lg = first_m2l_level();
  S.ng = group_level > 0 ? 1 << (3 * group_level) : 1;
  if (rc || (rc = mmax_buf.ensure(std::max<size_t>(MAXL + 1, (size_t)(lmax - lg + 1) * S.ng) * 4))) return rc;
  size_t off = 0;
  int wg = 0;
  for (int lev = l0; lev <= l1; lev++) {
    const int nb = si.nb[lev];
    if (nb == 0) continue;
    if (sj.nb[lev] == 0) {
      const long nl = (long)nb * P2 * 2;
      if (init) k_zero_t<float><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, lexp[lev].as<float>());
      continue;
    }
    S.M[S.nl] = mexp[lev].as<float>();
    S.Mh[S.nl] = mexp_h[lev].as<uint4>();
    S.mmax[S.nl] = mmax_buf.as<unsigned>() + (size_t)(lev - lg) * S.ng;
    S.key[S.nl] = sj.bkey[lev].as<uint32_t>();
    S.gs[S.nl] = group_shift(lev);
    S.off[S.nl + 1] = S.off[S.nl] + sj.nb[lev] + 1;
    const int ns = m2l_splits(lev);
    M2LLev& d = A.lv[A.nlv++] = m2l_desc(lev, 1, ORB_WPG, ns, m2l_part.as<float>() + off, init ? 1 : 0, wg);
    d.mmax = S.mmax[S.nl++];
    d.opH = hop_m2l.as<uint4>() + (size_t)(lev - 2) * NORBOP * frg;
    d.sa_e = hop_e[lev];
    wg += d.nwg;
    off += (size_t)ns * nb * rows;
  }
  if (A.nlv == 0) return FMMX_OK;
  if ((rc = launch_orbit_gen_order(p, S, stream))) return rc;
  if ((rc = launch_m2l_orbit_gen(p, A, wg, orbtab.as<int4>(), stream))) return rc;
  return launch_orbit_gen_reduce(p, A, stream);
}

// FP64 Laplace M2L of levels l0..l1 by reflection orbits, one launch; the locals
// are written (init) or added to
int Engine::run_m2l_f64(int l0, int l1, bool init) {
  M2LLaunch A{};
  MSplitLevels S{};
  const size_t rows = orbit_f64_rows(p);
  size_t need = 0;
  for (int lev = l0; lev <= l1; lev++)
    if (si.nb[lev] > 0 && sj.nb[lev] > 0) need += (size_t)m2l_splits(lev) * si.nb[lev] * rows;
  int rc = m2l_part.ensure(std::max<size_t>(need, 1) * 8);
  if (rc) return rc;
  size_t off = 0;
  int wg = 0;
  for (int lev = l0; lev <= l1; lev++) {
    const int nb = si.nb[lev];
    if (nb == 0) continue;
    if (sj.nb[lev] == 0) {
      const long nl = (long)nb * P2;
      if (init) k_zero_t<double><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, lexp[lev].as<double>());
      continue;
    }
    S.M[S.nl] = mexp[lev].as<float>();
    S.Mh[S.nl] = mexp_h[lev].as<uint4>();
    S.off[S.nl + 1] = S.off[S.nl] + sj.nb[lev] + 1;
    S.nl++;
    const int ns = m2l_splits(lev);
    float* part = reinterpret_cast<float*>(m2l_part.as<double>() + off);
    M2LLev& d = A.lv[A.nlv++] = m2l_desc(lev, 1, ORB_WPG, ns, part, init ? 1 : 0, wg);
    d.opH = op_m2l_of.as<uint4>();
    wg += d.nwg;
    off += (size_t)ns * nb * rows;
  }
  if (A.nlv == 0) return FMMX_OK;
  const bool tmark = per_phase && l1 == lmax;
  m2l_timed = m2l_timed || tmark;
  return launch_m2l_orbit_f64(p, S, A, wg, orbtab.as<int4>(), tmark ? ev[8] : nullptr, tmark ? ev[9] : nullptr, stream);
}

// phase 0: the M2L launch and (with splits) the reduction into the locals;
// 1: the launch alone, partial sums only (needs m2l_splits(lev) > 1);
// 2: the reduction alone, adding the partials of phase 1 to the locals
int Engine::run_m2l(int lev, bool init, int phase) {
  const int nb = si.nb[lev];
  if (nb == 0) return FMMX_OK;
  if (hh && !fp64) return run_m2l_hh(lev, lev, init);
  if (orbit_f64()) return run_m2l_f64(lev, lev, init);
  const long nl = (long)nb * P2 * parts();
  if (sj.nb[lev] == 0) {
    if (init && phase != 1) {
      if (fp64) k_zero_t<double><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, lexp[lev].as<double>());
      else k_zero_t<float><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, lexp[lev].as<float>());
    }
    return FMMX_OK;
  }
  const int MT = (P2 + 15) / 16, KS = (P2 + 3) / 4;
  // FP32: MFMA fragment order; FP64: k-major (transposed) operators
  const size_t FR = fp64 ? (size_t)P2 * P2 : (size_t)KS * MT * 64;
  const size_t opoff = (yk || m2l_per_level) ? (size_t)(lev - 2) * NOFF * FR : 0;
  DevBuf& opm2l = yk ? yop_m2l : op_m2l;
  const int tiles = (nb + M2L_TN - 1) / M2L_TN + 8;
  // enough workgroups to cover the chip: split the 189 offsets when tiles are few
  int nsplit = m2l_splits(lev);
  const size_t es = fp64 ? 8 : 4;
  if (phase == 2) {
    if (nsplit < 2) return fail(FMMX_ESTATE, "M2L reduction without partial sums");
    if (fp64)
      k_m2l_reduce<double><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, nsplit, part_buf->as<double>(),
                                                                        lexp[lev].as<double>(), init ? 1 : 0);
    else
      k_m2l_reduce<float><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, nsplit, part_buf->as<float>(),
                                                                       lexp[lev].as<float>(), init ? 1 : 0);
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  }
  if (phase == 1 && nsplit < 2) return fail(FMMX_ESTATE, "M2L partial sums need offset splits");
  const bool orbit = !fp64 && !hh && m2l_variant(lev).pa == 6;
  if (orbit && phase == 1) return fail(FMMX_ESTATE, "the orbit M2L reduces with its launch");
  if (nsplit > 1 || orbit) {
    int rc = part_buf->ensure(orbit ? (size_t)nsplit * nb * 8 * OLayout<2>::RW * es : (size_t)nsplit * nl * es);
    if (rc) return rc;
  }

  const int gsh = group_shift(lev);
  if (hh) {
    // FP64: split complex expansions, D = 2 p^2, k-major operators per level, on
    // the vector units
    const size_t hoff = (size_t)(lev - 2) * NOFF * 4 * P2 * P2;
    return dispatch_hp(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value;
      k_m2l_vec<P, double, 2><<<tiles * nsplit, 256, 0, stream>>>(
          lev, nb, nsplit, cls_cnt[lev].as<int>(), cls_ord[lev].as<uint32_t>(), si.bkey[lev].as<uint32_t>(),
          sj.dense[lev].as<int>(), mexp[lev].as<double>(), lexp[lev].as<double>(), part_buf->as<double>(),
          hop_m2l.as<double>() + hoff, offtab.as<int4>(), init ? 1 : 0, gsh, pair_ctr.as<unsigned long long>() + 2 + lev);
      if (nsplit > 1 && phase == 0)
        k_m2l_reduce<double><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, nsplit, part_buf->as<double>(),
                                                                          lexp[lev].as<double>(), init ? 1 : 0);
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  auto m2l = [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value;
    if (fp64) {
      const bool tmark = per_phase && lev == lmax;
      if (tmark) FMMX_HIP(hipEventRecord(ev[8], stream));
      k_m2l_vec<P, double><<<tiles * nsplit, 256, 0, stream>>>(
          lev, nb, nsplit, cls_cnt[lev].as<int>(), cls_ord[lev].as<uint32_t>(), si.bkey[lev].as<uint32_t>(),
          sj.dense[lev].as<int>(), mexp[lev].as<double>(), lexp[lev].as<double>(), part_buf->as<double>(),
          opm2l.as<double>() + opoff, offtab.as<int4>(), init ? 1 : 0, gsh, pair_ctr.as<unsigned long long>() + 2 + lev);
      if (tmark) {
        FMMX_HIP(hipEventRecord(ev[9], stream));
        m2l_timed = true;
      }
      if (nsplit > 1 && phase == 0)
        k_m2l_reduce<double><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, nsplit, part_buf->as<double>(),
                                                                          lexp[lev].as<double>(), init ? 1 : 0);
    } else if constexpr (P <= P_ALL) {
      const M2LVariant var = m2l_variant(lev);
      if (var.pa >= 3) {
        int r2 = upload_split(var.pa);
        if (r2) return r2;
      }
      M2LLaunch A{};
      A.nlv = 1;
      A.lv[0] = m2l_desc(lev, var.nt, var.wpg, nsplit, part_buf->as<float>(), init ? 1 : 0, 0);
      if (var.pa == 4) A.lv[0].offtab = offtab_s.as<int4>();
      if (var.pa == 5) {
        A.lv[0].offtab = offtab.as<int4>();
        A.lv[0].opH = op_m2l_w.as<uint4>();
      }
      if (orbit) A.lv[0].opH = op_m2l_o.as<uint4>();
      if (var.pa >= 3) {
        int r2 = run_msplit(lev, lev, var.pa);
        if (r2) return r2;
      }
      const bool tmark = per_phase && lev == lmax;
      if (tmark) FMMX_HIP(hipEventRecord(ev[8], stream));
      if (var.pa >= 3) {
        int r2 = orbit         ? launch_m2l_orbit(p, A, A.lv[0].nwg, orbtab.as<int4>(), stream)
                 : var.pa == 5 ? launch_m2l_wide(p, A, A.lv[0].nwg, var.wpg, var.nt, stream)
                               : launch_m2l_split(p, A, A.lv[0].nwg, var.nt, var.wpg, var.pa == 4, stream);
        if (r2) return r2;
      } else {
        launch_m2l<P>(A, A.lv[0].nwg, var.nt, var.pa, var.wpg, stream);
      }
      if (tmark) {
        FMMX_HIP(hipEventRecord(ev[9], stream));
        m2l_timed = true;
      }
      if (orbit) {
        int r2 = launch_orbit_reduce(p, A, stream);
        if (r2) return r2;
      } else if (nsplit > 1 && phase == 0) {
        k_m2l_reduce<float><<<(int)((nl + 255) / 256), 256, 0, stream>>>(nl, nsplit, part_buf->as<float>(),
                                                                         lexp[lev].as<float>(), init ? 1 : 0);
      }
    }
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  };
  return p > P_ALL ? dispatch_hi(p, m2l) : dispatch_p(p, m2l);
}

}  // namespace fmmx
