// translate.hip -- M2M and L2L (kernel/m2m.cxx, l2l.cxx) for CDNA4 (gfx950):
// dense p^2 x p^2 operators per child octant (level independent in the scaled
// basis), on MFMA in FP32 and, but for Helmholtz and order 18, in FP64.
#include "phases.h"

namespace fmmx {

namespace {

// ---------------------------------------------------------------------
// M2M and L2L as small batched GEMMs: a workgroup (128 threads) owns 16
// output boxes; per child octant the operator (VS x VS, k-major) is staged
// in LDS in K-chunks and applied to the 16 gathered input vectors, each
// thread holding a (rows x 4 boxes) register block.
//   M2M: output parent b, input = its child with octant o, summed over the
//        octants present (kernel/m2m.cxx:115-155).
//   L2L: the 16 children of a tile share one parity class, hence one octant
//        and one operator; output child = operator x its parent
//        (kernel/l2l.cxx:203-237).
constexpr int TR_TB = 16, TR_KC = 32, TR_BST = TR_TB + 4, TR_NT = 128;

template <int VS, typename T, int L2L>
__global__ __launch_bounds__(TR_NT) void k_translate(int nout, const int* __restrict__ cfirst,
                                                     const uint32_t* __restrict__ key, const int* __restrict__ parent,
                                                     const int* __restrict__ cls_cnt, const uint32_t* __restrict__ ord,
                                                     const T* __restrict__ in, T* __restrict__ out,
                                                     const T* __restrict__ opT) {
  // M2M: blockIdx.y = child octant; this block writes that octant's partial
  // product into out + octant * nout * VS (summed afterwards in fixed order)
  constexpr int RPT = (VS + 31) / 32, KC = VS > 160 ? TR_KC / 2 : TR_KC;  // LDS within 64 KB
  __shared__ T As[KC][VS];
  __shared__ T Bs[KC][TR_BST];
  __shared__ int src[TR_TB], dst[TR_TB];
  __shared__ int s_oct;
  const int tid = threadIdx.x;
  const int tx = tid & 3, ty = tid >> 2;  // 4 boxes x 32 row groups
  if (tid == 0) {
    int oct = -1;
    if (L2L) {
      // tile -> (class, index) over the class-sorted child list
      int t = blockIdx.x, start = 0;
      for (int c = 0; c < 8; c++) {
        const int cnt = cls_cnt[c], nt = (cnt + TR_TB - 1) / TR_TB;
        if (oct < 0 && t < nt) {
          // class bits (x,y,z) -> octant bits (y | x<<1 | z<<2)
          oct = ((c >> 1) & 1) | ((c & 1) << 1) | (c & 4);
          start += t * TR_TB;
          s_oct = oct;
          for (int k = 0; k < TR_TB; k++) {
            const int i = t * TR_TB + k;
            dst[k] = i < cnt ? (int)ord[start - t * TR_TB + i] : -1;
          }
        } else if (oct < 0) {
          t -= nt;
          start += cnt;
        }
      }
      if (oct < 0) s_oct = -1;
    } else {
      s_oct = 0;
      for (int k = 0; k < TR_TB; k++) {
        const int b = blockIdx.x * TR_TB + k;
        dst[k] = b < nout ? b : -1;
      }
    }
  }
  __syncthreads();
  if (s_oct < 0) return;
  T acc[RPT][4];
#pragma unroll
  for (int r = 0; r < RPT; r++)
#pragma unroll
    for (int c = 0; c < 4; c++) acc[r][c] = T(0);
  const int o_begin = L2L ? s_oct : (int)blockIdx.y, o_end = o_begin + 1;
  if (!L2L) out += (size_t)blockIdx.y * nout * VS;
  for (int o = o_begin; o < o_end; o++) {
    __syncthreads();
    if (tid < TR_TB) {
      const int b = dst[tid];
      int s = -1;
      if (b >= 0) {
        if (L2L) {
          s = parent[b];
        } else {
          for (int c = cfirst[b]; c < cfirst[b + 1]; c++)
            if ((int)(key[c] & 7) == o) s = c;
        }
      }
      src[tid] = s;
    }
    __syncthreads();
    const T* A = opT + (size_t)o * VS * VS;
    for (int k0 = 0; k0 < VS; k0 += KC) {
      const int kc = min(KC, VS - k0);
      __syncthreads();
      for (int e = tid; e < kc * VS; e += TR_NT) As[e / VS][e % VS] = A[(size_t)k0 * VS + e];
      for (int e = tid; e < kc * TR_TB; e += TR_NT) {
        const int t = e / kc, k = e % kc, s = src[t];
        Bs[k][t] = s >= 0 ? in[(size_t)s * VS + k0 + k] : T(0);
      }
      __syncthreads();
      for (int k = 0; k < kc; k++) {
        T bv[4];
#pragma unroll
        for (int c = 0; c < 4; c++) bv[c] = Bs[k][tx * 4 + c];
#pragma unroll
        for (int r = 0; r < RPT; r++) {
          const int row = ty + 32 * r;
          const T av = row < VS ? As[k][row] : T(0);
#pragma unroll
          for (int c = 0; c < 4; c++) acc[r][c] += av * bv[c];
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const int b = dst[tx * 4 + c];
    if (b < 0) continue;
#pragma unroll
    for (int r = 0; r < RPT; r++) {
      const int row = ty + 32 * r;
      if (row < VS) out[(size_t)b * VS + row] = acc[r][c];
    }
  }
}

// ---------------------------------------------------------------------
// M2M and L2L on MFMA (v_mfma_f32_16x16x4f32, v_mfma_f64_16x16x4f64), operators
// in the fragment order of the M2L kernel ([ks][mt][lane] holds row
// 16 mt + lane % 16, column (lane / 16) KS + ks of the p^2 x p^2 operator).
//   M2M: a workgroup of 8 waves owns 16 parent boxes; wave w multiplies the
//        octant-w operator with the 16 children of octant w (zero where a
//        parent has none) and the 8 products are summed in LDS in octant
//        order, so the result does not depend on scheduling
//        (kernel/m2m.cxx:115-155).
//   L2L: a wave owns 16 children of one parity class, which share one octant
//        and so one operator; each child's locals = operator x its parent's
//        (kernel/l2l.cxx:203-237).  The children's locals are written, or
//        added to when the level's M2L ran first (add).
// A box holds `parts` expansions side by side (2: the real and imaginary parts
// of the Helmholtz kernel, which one real operator carries alike: its regular
// re-expansions do not mix them); blockIdx.y is the part.  Helmholtz at p = 12
// on a sphere of 1M points (lmax 6), M2M and L2L of all levels: 1.41 + 1.15 ms
// as (2 p^2)^2 products on the vector units, 0.142 + 0.135 ms here.
// FP64 (the same fragments in double; a lane's output rows are 4 r + l / 16
// instead of 4 (l / 16) + r): 4,096 children at p = 10 24 + 23 us against 48 + 43
// us for one M2M and L2L level in k_translate, whose FMAs wait for LDS.
template <int P, int L2L, typename T>
__global__ __launch_bounds__(L2L ? 256 : 512) void k_translate_mfma(int nout, const int* __restrict__ cfirst,
                                                                    const uint32_t* __restrict__ key,
                                                                    const int* __restrict__ parent,
                                                                    const int* __restrict__ cls_cnt,
                                                                    const uint32_t* __restrict__ ord,
                                                                    const T* __restrict__ in,
                                                                    T* __restrict__ out,
                                                                    const T* __restrict__ opF, int add,
                                                                    int parts) {
  using ML = MLayout<P>;
  constexpr int P2 = P * P, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, FR = KS * MT * 64;
  using V4 = typename Mfma<T>::v4;
  constexpr bool D = sizeof(T) == 8;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, j = l & 15, kq = l >> 4;
  in += (size_t)blockIdx.y * (L2L ? P2 : ML::VS);
  out += (size_t)blockIdx.y * (L2L ? P2 : ML::VS);
  int dst = -1, src = -1, oct = 0;
  if (L2L) {
    // wave -> (class, tile) over the class-sorted child list
    int t = blockIdx.x * 4 + w, start = 0, c = 0;
    for (; c < 8; c++) {
      const int cnt = cls_cnt[c], nt = (cnt + 15) / 16;
      if (t < nt) break;
      t -= nt;
      start += cnt;
    }
    if (c == 8) return;  // no barrier below in this mode
    // class bits (x, y, z) -> octant bits (y | x << 1 | z << 2)
    oct = ((c >> 1) & 1) | ((c & 1) << 1) | (c & 4);
    const int i = t * 16 + j;
    if (i < cls_cnt[c]) {
      dst = (int)ord[start + i];
      src = parent[dst];
    }
  } else {
    oct = w;
    const int b = blockIdx.x * 16 + j;
    if (b < nout) {
      dst = b;
      for (int c = cfirst[b]; c < cfirst[b + 1]; c++)
        if ((int)(key[c] & 7) == oct) src = c;
    }
  }
  V4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++) acc[mt] = Mfma<T>::zero();
  if (__ballot(src >= 0) != 0) {
    T bv[KS];
    if (L2L) {
      const T* ps = in + (size_t)(src >= 0 ? src : 0) * parts * P2 + kq * KS;
#pragma unroll
      for (int ks = 0; ks < KS; ks++) bv[ks] = (src >= 0 && kq * KS + ks < P2) ? ps[ks] : T(0);
    } else {
      const V4* ms = reinterpret_cast<const V4*>(in + (size_t)(src >= 0 ? src : 0) * parts * ML::VS + kq * ML::KSP);
#pragma unroll
      for (int v4 = 0; v4 < ML::KSP / 4; v4++) {
        const V4 m4 = src >= 0 ? ms[v4] : V4{T(0), T(0), T(0), T(0)};
        if (4 * v4 + 0 < KS) bv[4 * v4 + 0] = (kq * KS + 4 * v4 + 0 < P2) ? m4[0] : T(0);
        if (4 * v4 + 1 < KS) bv[4 * v4 + 1] = (kq * KS + 4 * v4 + 1 < P2) ? m4[1] : T(0);
        if (4 * v4 + 2 < KS) bv[4 * v4 + 2] = (kq * KS + 4 * v4 + 2 < P2) ? m4[2] : T(0);
        if (4 * v4 + 3 < KS) bv[4 * v4 + 3] = (kq * KS + 4 * v4 + 3 < P2) ? m4[3] : T(0);
      }
    }
    const T* A = opF + (size_t)oct * FR + l;
#pragma unroll
    for (int ks = 0; ks < KS; ks++) {
      T af[MT];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) af[mt] = A[(ks * MT + mt) * 64];
#pragma unroll
      for (int mt = 0; mt < MT; mt++) acc[mt] = Mfma<T>::fma(af[mt], bv[ks], acc[mt]);
    }
  }
  if (L2L) {
    if (dst < 0) return;
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int i = 16 * mt + (D ? 4 * r + kq : 4 * kq + r);
        if (i < P2) {
          T* o = out + (size_t)dst * parts * P2 + i;
          *o = add ? *o + acc[mt][r] : acc[mt][r];
        }
      }
    return;
  }
  // M2M: the 8 octant products through LDS, summed in octant order
  __shared__ T red[8][MT * 4 * 64];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int r = 0; r < 4; r++) red[w][(mt * 4 + r) * 64 + l] = acc[mt][r];
  __syncthreads();
  for (int e = tid; e < 16 * ML::VS; e += 512) {
    const int jb = e / ML::VS, pos = e % ML::VS, b = blockIdx.x * 16 + jb;
    if (b >= nout) continue;
    // padded position -> slot (pads are written as zeros)
    const int seg = pos / ML::KSP, ks = pos % ML::KSP, i = seg * KS + ks;
    T v = T(0);
    if (ks < KS && i < P2) {
      const int lo = i & 3, hi = (i >> 2) & 3;
      const int q = ((i >> 4) * 4 + (D ? hi : lo)) * 64 + (D ? lo : hi) * 16 + jb;
#pragma unroll
      for (int o = 0; o < 8; o++) v += red[o][q];
    }
    out[(size_t)b * parts * ML::VS + pos] = v;
  }
}

}  // namespace

int Engine::run_m2m(int lev) {
  const int nbp = sj.nb[lev];
  if (nbp == 0) return FMMX_OK;
  if (!fp64 || (!hh && p <= P_ALL)) {
    return dispatch_p(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value;
      auto go = [&](auto t) {
        using T = typename decltype(t)::type;
        k_translate_mfma<P, 0, T><<<dim3((nbp + 15) / 16, parts()), 512, 0, stream>>>(
            nbp, sj.cfirst[lev].as<int>(), sj.bkey[lev + 1].as<uint32_t>(), nullptr, nullptr, nullptr,
            mexp[lev + 1].as<T>(), mexp[lev].as<T>(), m2m_ops<T>(lev), 0, parts());
      };
      if (fp64) go(tag<double>{});
      else go(tag<float>{});
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  // FP64 Helmholtz and the order above P_ALL: vector units
  const dim3 grid((nbp + TR_TB - 1) / TR_TB, 8);
  const long n = (long)nbp * VS * parts();
  int rc = m2m_part.ensure((size_t)8 * n * 8);
  if (rc) return rc;
  if (hh) {
    return dispatch_hp(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value, V = 2 * MLayout<P>::VS;
      k_translate<V, double, 0><<<grid, TR_NT, 0, stream>>>(
          nbp, sj.cfirst[lev].as<int>(), sj.bkey[lev + 1].as<uint32_t>(), nullptr, nullptr, nullptr,
          mexp[lev + 1].as<double>(), m2m_part.as<double>(), m2m_ops<double>(lev));
      k_m2l_reduce<double><<<(int)((n + 255) / 256), 256, 0, stream>>>(n, 8, m2m_part.as<double>(),
                                                                       mexp[lev].as<double>(), 1);
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  auto m2m = [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value, V = MLayout<P>::VS;
    k_translate<V, double, 0><<<grid, TR_NT, 0, stream>>>(
        nbp, sj.cfirst[lev].as<int>(), sj.bkey[lev + 1].as<uint32_t>(), nullptr, nullptr, nullptr,
        mexp[lev + 1].as<double>(), m2m_part.as<double>(), m2m_ops<double>(lev));
    k_m2l_reduce<double><<<(int)((n + 255) / 256), 256, 0, stream>>>(n, 8, m2m_part.as<double>(),
                                                                     mexp[lev].as<double>(), 1);
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  };
  return dispatch_hi(p, m2m);
}

int Engine::run_l2l(int lev, bool add) {
  const int nbc = si.nb[lev];
  if (nbc == 0) return FMMX_OK;
  if (!fp64 || (!hh && p <= P_ALL)) {
    // one wave per 16 children of a class: at most nbc / 16 + 8 waves
    return dispatch_p(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value;
      auto go = [&](auto t) {
        using T = typename decltype(t)::type;
        k_translate_mfma<P, 1, T><<<dim3((nbc / 16 + 8 + 3) / 4, parts()), 256, 0, stream>>>(
            nbc, nullptr, nullptr, si.parent[lev].as<int>(), cls_cnt[lev].as<int>(), cls_ord[lev].as<uint32_t>(),
            lexp[lev - 1].as<T>(), lexp[lev].as<T>(), l2l_ops<T>(lev), add ? 1 : 0, parts());
      };
      if (fp64) go(tag<double>{});
      else go(tag<float>{});
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  if (add) return fail(FMMX_ESTATE, "the L2L add form is on MFMA only");
  const int grid = (nbc + TR_TB - 1) / TR_TB + 8;
  if (hh) {
    return dispatch_hp(p, [&](auto pc) -> int {
      constexpr int P = decltype(pc)::value, Q = 2 * P * P;
      k_translate<Q, double, 1><<<grid, TR_NT, 0, stream>>>(
            nbc, nullptr, si.bkey[lev].as<uint32_t>(), si.parent[lev].as<int>(), cls_cnt[lev].as<int>(),
            cls_ord[lev].as<uint32_t>(), lexp[lev - 1].as<double>(), lexp[lev].as<double>(), l2l_ops<double>(lev));
      FMMX_HIP(hipGetLastError());
      return FMMX_OK;
    });
  }
  auto l2l = [&](auto pc) -> int {
    constexpr int P = decltype(pc)::value, Q = P * P;
    k_translate<Q, double, 1><<<grid, TR_NT, 0, stream>>>(
          nbc, nullptr, si.bkey[lev].as<uint32_t>(), si.parent[lev].as<int>(), cls_cnt[lev].as<int>(),
          cls_ord[lev].as<uint32_t>(), lexp[lev - 1].as<double>(), lexp[lev].as<double>(), l2l_ops<double>(lev));
    FMMX_HIP(hipGetLastError());
    return FMMX_OK;
  };
  return dispatch_hi(p, l2l);
}

}  // namespace fmmx
