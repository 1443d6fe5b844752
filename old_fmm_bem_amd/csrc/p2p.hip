// p2p.hip -- near field and direct sums for CDNA4 (gfx950), wave64.
//   P2P  kernel/G_p2p.cxx, Gni_p2p.cxx, Gnj_p2p.cxx: work items of a target
//        leaf box (two or more lanes per target for small leaves), source particles
//        of the near boxes staged through LDS, FP32 (or FP64) pair math, FP64
//        per-target sums.
//   direct sums kernel/G_dir.cxx, Gni_dir.cxx, Gnj_dir.cxx.
#include "phases.h"

namespace fmmx {

namespace {

// ---------------------------------------------------------------------
// reciprocal square root: v_rsq_f32 (1 ulp) in FP32, full precision in FP64
__device__ __forceinline__ float rsq(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq(double x) { return rsqrt(x); }
__device__ __forceinline__ float yexp(float x) { return __expf(x); }
__device__ __forceinline__ double yexp(double x) { return exp(x); }

// ---------------------------------------------------------------------
// P2P: a workgroup per work item (up to BS targets of a leaf box), sources of
// each near box staged through LDS in tiles of BS.
//
// A staged source: in doubles where the pair computes in them (FP64, EXACT), so
// that the four conversions, exact either way, are paid once per staging and
// not once per pair; REF subtracts in float
// (250,000 points, lmax 4: 0.47 -> 0.44 ms; a direct sum of 2,000 targets by
// 300,000 sources 0.89 -> 0.85 ms).
struct alignas(32) SrcD {
  double x, y, z, w;
};
template <typename T, int CONV>
using Src = std::conditional_t<sizeof(T) == 8 && CONV == FMMX_CONV_EXACT, SrcD, float4>;

template <typename T, int NEQ, int CONV, bool SELF = true>
__device__ __forceinline__ void pair(float xi, float yi, float zi, float nxi, float nyi, float nzi,
                                     Src<T, CONV> s, float4 sn, T& p, T& fx, T& fy, T& fz, T lam = T(0)) {
  T dx, dy, dz;
  if (CONV == FMMX_CONV_REF || sizeof(T) == 4) {
    dx = T(xi - s.x);  // float subtraction as kernel/G_p2p.cxx:21-23
    dy = T(yi - s.y);
    dz = T(zi - s.z);
  } else {
    dx = T(xi) - T(s.x);
    dy = T(yi) - T(s.y);
    dz = T(zi) - T(s.z);
  }
  T r2 = dx * dx + dy * dy + dz * dz;
  T inv;
  if (CONV == FMMX_CONV_REF) {
    r2 += T(EPSF);
    inv = rsq(r2);
  } else {
    inv = rsq(r2);
    if (SELF) inv = r2 > T(0) ? inv : T(0);  // coincident pair excluded (select, no branch)
  }
  const T qi = T(s.w) * inv;
  if (NEQ == FMMX_HELMHOLTZ) {
    // (qr + i qi) exp(i k r) / r: real part into p, imaginary part into fx
    // (sn.x carries the imaginary part of the charge, lam the wavenumber)
    const T r = r2 * inv;
    T sk, ck;
    if constexpr (sizeof(T) == 4) {
      // hardware sine/cosine (argument in revolutions): near-field k r is
      // O(1), where their absolute error is far below the FP32 path's
      const float t = float(lam * r) * 0.15915494309189535f;
      sk = __builtin_amdgcn_sinf(t);
      ck = __builtin_amdgcn_cosf(t);
    } else {
      sincos(lam * r, &sk, &ck);
    }
    const T qim = T(sn.x) * inv;
    p += qi * ck - qim * sk;
    fx += qi * sk + qim * ck;
  } else if (NEQ == FMMX_YUKAWA) {
    // exp(-lambda r)/r (kernel/Helmholtz_G_p2p.cxx:22 without its constant
    // (pi/2)/lambda); gradient -(1 + lambda r) e d / r^3
    const T r = r2 * inv;
    const T e = qi * yexp(-lam * r);
    p += e;
    const T rs = e * (T(1) + lam * r) * inv * inv;
    fx -= dx * rs;
    fy -= dy * rs;
    fz -= dz * rs;
  } else if (NEQ == FMMX_G) {
    p += qi;
    const T rs = qi * inv * inv;
    fx -= dx * rs;
    fy -= dy * rs;
    fz -= dz * rs;
  } else if (NEQ == FMMX_GNI) {
    p += (dx * T(nxi) + dy * T(nyi) + dz * T(nzi)) * (qi * inv * inv);
  } else {
    p += (dx * T(sn.x) + dy * T(sn.y) + dz * T(sn.z)) * (qi * inv * inv);
  }
}

// TPT lanes per target (2: leaves of at most about 32 targets, one wave per
// workgroup): the lanes of a target take alternating staged sources and add
// their sums at the end, so a half-empty leaf does not idle half the wave.
// With TPT 2 each item picks its own lanes per target (2, 4, 8 or 16) from the
// targets it has, so an item of a few targets (a leaf of 10, the rest of one of
// 33-40) still keeps the wave's lanes busy.
//
// A workgroup takes work items, each a leaf and up to `tmax` of its targets
// (k_p2p_items), so that a leaf of many targets is spread over the chip: 60,000
// points in 64 leaves (lmax 2, REF) 4.13 -> 0.71 ms against one workgroup per
// leaf; a Plummer cloud of 120,000 targets whose core leaves hold over 100
// (lmax 7) 0.31 -> 0.14 ms.  With 32 targets per item the sums are those of
// one workgroup per leaf in 32-target passes, bit for bit.

// Shape of the near field for n targets in nb leaves: the one-wave form (lanes
// per target chosen per item) or `lanes` lanes, one per target, and targets per
// item.  One wave for leaves of at most `small` targets on average (measured
// 36-47% less P2P time than one lane per target in 64/128-lane blocks at 46-61
// targets per leaf; 256-lane blocks win above 96: 2.95 against 3.55 ms at 244
// per leaf), and for every leaf size while 256-target blocks would leave the
// chip idle.  Its items hold 32 targets (two lanes each), fewer where that
// leaves the 1,024 SIMDs fewer than two waves each (1,000 points in 64 leaves:
// 4 per item), and a quarter of that in leaves of over `heavy` targets, so that
// an item's work (targets x sources) stays within a few times the others'.
struct P2PShape {
  int one_wave, lanes, tmax, heavy;
};
__host__ __device__ inline P2PShape p2p_shape(int n, int nb, double small, bool fixed) {
  const double mean = (double)n / (nb > 0 ? nb : 1);
  P2PShape s{};
  s.one_wave = mean <= small || (!fixed && n / 256 + nb / 2 < 1024);
  s.lanes = s.one_wave ? 64 : mean > 96 ? 256 : mean > 40 ? 128 : 64;
  s.tmax = s.one_wave ? 32 : s.lanes;
  if (s.one_wave)
    while (s.tmax > 4 && n / s.tmax + nb < 2048) s.tmax /= 2;
  s.heavy = !s.one_wave || mean > 1e8 ? 1 << 30 : mean > 16 ? (int)(4 * mean) : 64;
  return s;
}
__device__ __forceinline__ int p2p_targets(int n, const P2PShape& s) {
  return n <= s.heavy ? s.tmax : s.tmax > 8 ? s.tmax / 4 : s.tmax;
}
// items of all leaves (their number is read on the device: the launch precedes
// the host's readback of it)
__global__ __launch_bounds__(256) void k_p2p_items(int n_, const int* __restrict__ nb_, double small, int fixed,
                                                   const int* __restrict__ first, const int* __restrict__ last,
                                                   int2* __restrict__ items, int* __restrict__ count) {
  const int nbi = *nb_;
  const P2PShape sh = p2p_shape(n_, nbi, small, fixed != 0);
  const int b = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63;
  int i0 = 0, n = 0, t = 1, c = 0;
  if (b < nbi) {
    i0 = first[b];
    n = last[b] - i0 + 1;
    t = p2p_targets(n, sh);
    c = (n + t - 1) / t;
  }
  int s = c;  // inclusive sums over the wave: one atomic per wave
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(s, d);
    if (lane >= d) s += u;
  }
  int base = 0;
  if (lane == 63 && s > 0) base = atomicAdd(count, s);
  base = __shfl(base, 63) + s - c;
  for (int k = 0; k < c; k++) items[base + k] = make_int2(b, i0 + k * t);
}

template <typename T, int NEQ, int CONV, int BS, int TPT = 1>
__global__ __launch_bounds__(BS) void k_p2p(const int2* __restrict__ items, const int* __restrict__ nitems, P2PShape shape,
                                            const uint32_t* __restrict__ ikey, const uint32_t* __restrict__ jkey,
                                            const int* __restrict__ ifirst, const int* __restrict__ ilast,
                                            const int* __restrict__ nij, const int* __restrict__ neij,
                                            const int* __restrict__ jfirst, const int* __restrict__ jlast,
                                            const float* __restrict__ xi, const float* __restrict__ yi,
                                            const float* __restrict__ zi, const float* __restrict__ nxi,
                                            const float* __restrict__ nyi, const float* __restrict__ nzi,
                                            const float* __restrict__ xj, const float* __restrict__ yj,
                                            const float* __restrict__ zj, const float* __restrict__ q,
                                            const float* __restrict__ nxj, const float* __restrict__ nyj,
                                            const float* __restrict__ nzj, double c4, double* __restrict__ vs,
                                            double* __restrict__ gxs, double* __restrict__ gys,
                                            double* __restrict__ gzs, double lamd) {
  constexpr bool GRAD = NEQ == FMMX_G || NEQ == FMMX_YUKAWA;
  // Helmholtz: nxj holds the imaginary parts of the charges, gxs receives the
  // imaginary part of the potential
  constexpr bool HH = NEQ == FMMX_HELMHOLTZ, SN = NEQ == FMMX_GNJ || HH;
  const T lam = T(lamd);
  // staging slots (SB = SPT x BS, each thread stages SPT of them) and near
  // boxes packed per round: the one-wave form stages up to 256 sources of up
  // to 8 boxes, so a leaf's 27 near boxes take a few rounds instead of ~14
  constexpr int SPT = TPT == 2 ? 4 : 1, SB = SPT * BS, KB = TPT == 2 ? 8 : 4;
  using S4 = Src<T, CONV>;
  __shared__ S4 sp[SB];
  __shared__ float4 sn[SN ? SB : 1];
  static_assert(TPT == 1 || (TPT == 2 && BS == 64), "two lanes per target within one wave");
  const int tid = threadIdx.x, ni = *nitems;
  for (int it = blockIdx.x; it < ni; it += gridDim.x) {
    const int2 item = items[it];
    const int b = item.x, base = item.y, nn = nij[b];
    const int i1 = min(ilast[b], base + p2p_targets(ilast[b] - ifirst[b] + 1, shape) - 1);
    // lanes per target (uniform): TPT, or up to 16 (TPT 2) for few targets
    int tpt = TPT;
    if (TPT == 2) {
      const int m = i1 - base + 1;
      tpt = m > 16 ? 2 : m > 8 ? 4 : m > 4 ? 8 : 16;
    }
    const int tb = BS / tpt;  // targets the lanes cover
    const int tt = tid % tb, part = tid / tb;
    const int i = base + tt;
    const bool act = i <= i1;
    float px = 0, py = 0, pz = 0, qx = 0, qy = 0, qz = 0;
    if (act) {
      px = xi[i];
      py = yi[i];
      pz = zi[i];
      if (NEQ == FMMX_GNI) {
        qx = nxi[i];
        qy = nyi[i];
        qz = nzi[i];
      }
    }
    double ap = 0, ax = 0, ay = 0, az = 0;
    const uint32_t kb = ikey[b];
    for (int e = 0; e < nn;) {
      // one staging round: near boxes e .. e + nbox - 1 packed into the SB
      // slots when they fit together (fewer barriers and shorter tails for
      // small leaves), else box e's sources SB at a time.  The target's own
      // box keeps a round to itself: only its pairs need the coincident test
      int jj = neij[b * NNEAR + e];
      int j0 = jfirst[jj], j1 = jlast[jj];
      int nbox = 1, cnt0 = j1 - j0 + 1, tot = cnt0;
      int s0[KB], c0[KB];
      s0[0] = j0;
      c0[0] = cnt0;
      const bool self = jkey[jj] == kb;
      bool packing = cnt0 <= SB && !self;
#pragma unroll
      for (int k = 1; k < KB; k++) {
        s0[k] = 0;
        c0[k] = 0;
        if (packing && e + k < nn) {
          const int jn = neij[b * NNEAR + e + k];
          const int a0 = jfirst[jn], c = jlast[jn] - a0 + 1;
          if (tot + c <= SB && jkey[jn] != kb) {
            s0[k] = a0;
            c0[k] = c;
            tot += c;
            nbox = k + 1;
          } else {
            packing = false;
          }
        }
      }
      const int rounds = cnt0 <= SB ? 1 : (cnt0 + SB - 1) / SB;
      for (int rr = 0; rr < rounds; rr++) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < SPT; u++) {
          const int slot = tid + u * BS;
          int js = -1;
          if (cnt0 <= SB) {
            // slot -> (packed box, offset)
            int t = slot;
#pragma unroll
            for (int k = 0; k < KB; k++) {
              if (js < 0 && k < nbox) {
                if (t < c0[k]) js = s0[k] + t;
                else t -= c0[k];
              }
            }
          } else if (rr * SB + slot < cnt0) {
            js = j0 + rr * SB + slot;
          }
          if (js >= 0) {
            sp[slot] = S4{xj[js], yj[js], zj[js], q[js]};
            if (NEQ == FMMX_GNJ) sn[slot] = make_float4(nxj[js], nyj[js], nzj[js], 0.f);
            if (HH) sn[slot] = make_float4(nxj[js], 0.f, 0.f, 0.f);
          }
        }
        __syncthreads();
        const int cnt = cnt0 <= SB ? tot : min(SB, cnt0 - rr * SB);
        T p = T(0), fx = T(0), fy = T(0), fz = T(0);
        // staged sources part, part + L, part + 2L, ... of the L lanes of a
        // target (L a compile-time stride: LDS offsets stay immediates)
        auto sweep = [&](auto lc) {
          constexpr int L = decltype(lc)::value;
          int s = part;
          // coincident points can only share a box key; other box pairs skip the test
          if (CONV == FMMX_CONV_EXACT && !self) {
            for (; s + 3 * L < cnt; s += 4 * L) {
#pragma unroll
              for (int u = 0; u < 4; u++)
                pair<T, NEQ, CONV, false>(px, py, pz, qx, qy, qz, sp[s + u * L], sn[SN ? s + u * L : 0], p, fx,
                                          fy, fz, lam);
            }
            for (; s < cnt; s += L)
              pair<T, NEQ, CONV, false>(px, py, pz, qx, qy, qz, sp[s], sn[SN ? s : 0], p, fx, fy, fz, lam);
          } else {
            for (; s + 3 * L < cnt; s += 4 * L) {
#pragma unroll
              for (int u = 0; u < 4; u++)
                pair<T, NEQ, CONV>(px, py, pz, qx, qy, qz, sp[s + u * L], sn[SN ? s + u * L : 0], p, fx, fy,
                                   fz, lam);
            }
            for (; s < cnt; s += L)
              pair<T, NEQ, CONV>(px, py, pz, qx, qy, qz, sp[s], sn[SN ? s : 0], p, fx, fy, fz, lam);
          }
        };
        if constexpr (TPT == 1) {
          sweep(std::integral_constant<int, 1>{});
        } else {
          if (tpt == 2) sweep(std::integral_constant<int, 2>{});
          else if (tpt == 4) sweep(std::integral_constant<int, 4>{});
          else if (tpt == 8) sweep(std::integral_constant<int, 8>{});
          else sweep(std::integral_constant<int, 16>{});
        }
        ap += (double)p;
        if (GRAD || HH) {
          ax += (double)fx;
          ay += (double)fy;
          az += (double)fz;
        }
      }
      e += nbox;
    }
    if (TPT == 2) {
      // the lanes of a target are tt, tt + tb, tt + 2 tb, ... of the one
      // wave: butterfly over the lane bits at and above tb (fixed order)
      for (int d = tb; d < 64; d <<= 1) {
        ap += __shfl_xor(ap, d, 64);
        if (GRAD || HH) {
          ax += __shfl_xor(ax, d, 64);
          ay += __shfl_xor(ay, d, 64);
          az += __shfl_xor(az, d, 64);
        }
      }
    }
    if (act && part == 0) {
      vs[i] = c4 * ap;
      if (HH) gxs[i] = c4 * ax;
      if (GRAD) {
        gxs[i] = c4 * ax;
        gys[i] = c4 * ay;
        gzs[i] = c4 * az;
      }
    }
  }
}

// direct sums: block of 64 targets x a slice of the sources, FP64 pair math,
// partial sums combined with atomics (outputs zeroed first)
template <int NEQ, int CONV>
__global__ __launch_bounds__(64) void k_direct(int ni, const float* __restrict__ xi, const float* __restrict__ yi,
                                               const float* __restrict__ zi, const float* __restrict__ nxi,
                                               const float* __restrict__ nyi, const float* __restrict__ nzi, int nj,
                                               const float* __restrict__ xj, const float* __restrict__ yj,
                                               const float* __restrict__ zj, const float* __restrict__ q,
                                               const float* __restrict__ nxj, const float* __restrict__ nyj,
                                               const float* __restrict__ nzj, int slice, double c4,
                                               double* __restrict__ v, double* __restrict__ gx,
                                               double* __restrict__ gy, double* __restrict__ gz, double lam) {
  constexpr bool GRAD = NEQ == FMMX_G || NEQ == FMMX_YUKAWA, HH = NEQ == FMMX_HELMHOLTZ;
  using S4 = Src<double, CONV>;
  __shared__ S4 sp[64];
  __shared__ float4 sn[64];
  const int i = blockIdx.x * 64 + threadIdx.x;
  const bool act = i < ni;
  float px = 0, py = 0, pz = 0, qx = 0, qy = 0, qz = 0;
  if (act) {
    px = xi[i];
    py = yi[i];
    pz = zi[i];
    if (NEQ == FMMX_GNI) {
      qx = nxi[i];
      qy = nyi[i];
      qz = nzi[i];
    }
  }
  const int j0 = blockIdx.y * slice, j1 = min(nj, j0 + slice);
  double p = 0, fx = 0, fy = 0, fz = 0;
  for (int jb = j0; jb < j1; jb += 64) {
    const int js = jb + threadIdx.x;
    __syncthreads();
    if (js < j1) {
      sp[threadIdx.x] = S4{xj[js], yj[js], zj[js], q[js]};
      if (NEQ == FMMX_GNJ) sn[threadIdx.x] = make_float4(nxj[js], nyj[js], nzj[js], 0.f);
      if (HH) sn[threadIdx.x] = make_float4(nxj[js], 0.f, 0.f, 0.f);  // imaginary charge
    }
    __syncthreads();
    const int cnt = min(64, j1 - jb);
#pragma unroll 4
    for (int s = 0; s < cnt; s++)
      pair<double, NEQ, CONV>(px, py, pz, qx, qy, qz, sp[s], sn[s], p, fx, fy, fz, lam);
  }
  if (act) {
    atomicAdd(&v[i], c4 * p);
    if (HH) atomicAdd(&gx[i], c4 * fx);
    if (GRAD) {
      atomicAdd(&gx[i], c4 * fx);
      atomicAdd(&gy[i], c4 * fy);
      atomicAdd(&gz[i], c4 * fz);
    }
  }
}

__global__ void k_zero_d(long n, double* __restrict__ a) {
  long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = 0;
}

}  // namespace

namespace {
__global__ void k_zero_i(int* a) {
  if (threadIdx.x == 0) *a = 0;
}
constexpr double P2P_SMALL = 96.0;  // FMMX_P2P_SMALL sets the bound instead
}  // namespace

// The work items of the tree in use (p2p_count cleared before); box counts may
// still be on the device only
int Engine::build_p2p_items() {
  const int n = si.n;
  if (n == 0) return FMMX_OK;
  const char* es = getenv("FMMX_P2P_SMALL");
  p2p_bound[0] = es ? atof(es) : P2P_SMALL;
  p2p_bound[1] = es ? 1.0 : 0.0;
  const long nbmax = std::min<long>(n, 1L << (3 * lmax));
  int rc = p2p_items.ensure(((size_t)nbmax + n / 4 + 1) * 8);
  if (rc) return rc;
  k_p2p_items<<<(int)((nbmax + 255) / 256), 256, 0, stream>>>(n, si.cnt.as<int>() + lmax, p2p_bound[0],
                                                              p2p_bound[1] != 0, si.bfirst[lmax].as<int>(),
                                                              si.blast.as<int>(), p2p_items.as<int2>(),
                                                              p2p_count.as<int>());
  FMMX_HIP(hipGetLastError());
  return FMMX_OK;
}

int Engine::run_p2p(int neq) {
  const int nbi = si.nb[lmax];
  if (nbi == 0) return FMMX_OK;
  const double cc = neq == FMMX_YUKAWA ? c_yukawa() : c4();
  const bool ref = cfg.convention == FMMX_CONV_REF;
  // Helmholtz: the imaginary charges ride in the source-normal slot, k in lambda's
  const float* nxj = neq == FMMX_HELMHOLTZ ? qs2.as<float>() : sj.nx.as<float>();
  const double kl = neq == FMMX_HELMHOLTZ ? hk : lam;
  const char* es = getenv("FMMX_P2P_SMALL");
  const P2PShape shape = p2p_shape(si.n, nbi, es ? atof(es) : P2P_SMALL, es != nullptr);
  const double now[2] = {es ? atof(es) : P2P_SMALL, es ? 1.0 : 0.0};
  int rc = FMMX_OK;
  if (now[0] != p2p_bound[0] || now[1] != p2p_bound[1]) {
    // the bound changed since the items were built (a captured evaluation's
    // launches keep theirs)
    p2p_items.renew();
    p2p_count.renew();
    if ((rc = p2p_count.ensure(4))) return rc;
    k_zero_i<<<1, 64, 0, stream>>>(p2p_count.as<int>());
    if ((rc = build_p2p_items())) return rc;
  }
  // about the number of items (known on the device); each workgroup strides
  const int grid = nbi + si.n / (2 * shape.tmax) + 1;
  auto go = [&](auto tag_t, auto neq_c, auto conv_c, auto bs_c, auto tpt_c) -> int {
    using T = typename decltype(tag_t)::type;
    constexpr int NEQ = decltype(neq_c)::value, CONV = decltype(conv_c)::value, BS = decltype(bs_c)::value;
    constexpr int TPT = decltype(tpt_c)::value;
    k_p2p<T, NEQ, CONV, BS, TPT><<<grid, BS, 0, stream>>>(
        p2p_items.as<int2>(), p2p_count.as<int>(), shape, si.bkey[lmax].as<uint32_t>(), sj.bkey[lmax].as<uint32_t>(), si.bfirst[lmax].as<int>(), si.blast.as<int>(), nij.as<int>(), neij.as<int>(), sj.bfirst[lmax].as<int>(),
        sj.blast.as<int>(), si.x.as<float>(), si.y.as<float>(), si.z.as<float>(), si.nx.as<float>(), si.ny.as<float>(),
        si.nz.as<float>(), sj.x.as<float>(), sj.y.as<float>(), sj.z.as<float>(), qs.as<float>(), nxj,
        sj.ny.as<float>(), sj.nz.as<float>(), cc, vs.as<double>(), gxs.as<double>(), gys.as<double>(),
        gzs.as<double>(), kl);
    return FMMX_OK;
  };
  auto by_bs = [&](auto t, auto nq, auto cv) -> int {
    using one = std::integral_constant<int, 1>;
    if (shape.one_wave) return go(t, nq, cv, std::integral_constant<int, 64>{}, std::integral_constant<int, 2>{});
    if (shape.lanes == 256) return go(t, nq, cv, std::integral_constant<int, 256>{}, one{});
    if (shape.lanes == 128) return go(t, nq, cv, std::integral_constant<int, 128>{}, one{});
    return go(t, nq, cv, std::integral_constant<int, 64>{}, one{});
  };
  auto by_conv = [&](auto t, auto nq) -> int {
    return ref ? by_bs(t, nq, std::integral_constant<int, FMMX_CONV_REF>{})
               : by_bs(t, nq, std::integral_constant<int, FMMX_CONV_EXACT>{});
  };
  auto by_neq = [&](auto t) -> int {
    if (neq == FMMX_HELMHOLTZ) return by_conv(t, std::integral_constant<int, FMMX_HELMHOLTZ>{});
    if (neq == FMMX_YUKAWA) return by_conv(t, std::integral_constant<int, FMMX_YUKAWA>{});
    if (neq == FMMX_G) return by_conv(t, std::integral_constant<int, FMMX_G>{});
    if (neq == FMMX_GNI) return by_conv(t, std::integral_constant<int, FMMX_GNI>{});
    return by_conv(t, std::integral_constant<int, FMMX_GNJ>{});
  };
  rc = fp64 ? by_neq(tag<double>{}) : by_neq(tag<float>{});
  if (rc) return rc;
  FMMX_HIP(hipGetLastError());
  return FMMX_OK;
}

int Engine::run_direct(int neq, int ni, const float* xi, const float* yi, const float* zi, const float* nxi,
                       const float* nyi, const float* nzi, int nj, const float* xj, const float* yj, const float* zj,
                       const float* nxj, const float* nyj, const float* nzj, const float* qj, double* v, double* gx,
                       double* gy, double* gz) {
  if (ni == 0) return FMMX_OK;
  long nz4 = ni;
  k_zero_d<<<(int)((nz4 + 255) / 256), 256, 0, stream>>>(nz4, v);
  if (neq == FMMX_HELMHOLTZ) k_zero_d<<<(int)((nz4 + 255) / 256), 256, 0, stream>>>(nz4, gx);  // Im part
  if (neq == FMMX_G || neq == FMMX_YUKAWA) {
    k_zero_d<<<(int)((nz4 + 255) / 256), 256, 0, stream>>>(nz4, gx);
    k_zero_d<<<(int)((nz4 + 255) / 256), 256, 0, stream>>>(nz4, gy);
    k_zero_d<<<(int)((nz4 + 255) / 256), 256, 0, stream>>>(nz4, gz);
  }
  if (nj == 0) return FMMX_OK;
  const int tb = (ni + 63) / 64;
  // 8 waves per SIMD hide the reciprocal root's chain (2,000 targets by 300,000
  // sources: 0.856 ms with 2 waves, 0.674 with 4, 0.544 with 8, 0.542 with 12),
  // in slices of at least 256 sources where 2 waves per SIMD leave that much
  // (each slice ends with its targets' atomics)
  const int ns2 = 2048 / tb, ns8 = 8192 / tb;
  int ns = std::max(1, std::min(1024, std::max(ns2, std::min(ns8, nj / 256))));
  int slice = (nj + ns - 1) / ns;
  slice = ((slice + 63) / 64) * 64;
  ns = (nj + slice - 1) / slice;
  dim3 grid(tb, ns);
  const bool ref = cfg.convention == FMMX_CONV_REF;
  const double cc = neq == FMMX_YUKAWA ? c_yukawa() : c4();
  // Helmholtz: nxj carries the imaginary charges, gx receives Im of the potential
  const double kl = neq == FMMX_HELMHOLTZ ? hk : lam;
#define FMMX_DIR(NEQ, CONV)                                                                                      \
  k_direct<NEQ, CONV><<<grid, 64, 0, stream>>>(ni, xi, yi, zi, nxi, nyi, nzi, nj, xj, yj, zj, qj, nxj, nyj, nzj, \
                                               slice, cc, v, gx, gy, gz, kl)
  if (neq == FMMX_HELMHOLTZ) {
    if (ref) FMMX_DIR(FMMX_HELMHOLTZ, FMMX_CONV_REF);
    else FMMX_DIR(FMMX_HELMHOLTZ, FMMX_CONV_EXACT);
  } else if (neq == FMMX_YUKAWA) {
    if (ref) FMMX_DIR(FMMX_YUKAWA, FMMX_CONV_REF);
    else FMMX_DIR(FMMX_YUKAWA, FMMX_CONV_EXACT);
  } else if (ref) {
    if (neq == FMMX_G) FMMX_DIR(FMMX_G, FMMX_CONV_REF);
    else if (neq == FMMX_GNI) FMMX_DIR(FMMX_GNI, FMMX_CONV_REF);
    else FMMX_DIR(FMMX_GNJ, FMMX_CONV_REF);
  } else {
    if (neq == FMMX_G) FMMX_DIR(FMMX_G, FMMX_CONV_EXACT);
    else if (neq == FMMX_GNI) FMMX_DIR(FMMX_GNI, FMMX_CONV_EXACT);
    else FMMX_DIR(FMMX_GNJ, FMMX_CONV_EXACT);
  }
#undef FMMX_DIR
  FMMX_HIP(hipGetLastError());
  return FMMX_OK;
}

}  // namespace fmmx
