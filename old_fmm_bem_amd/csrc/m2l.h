// m2l.h -- expansion layouts, reflection signs and launch descriptors shared
// by the M2L kernels (m2l.hip: FP32 and FP64 forms; m2l_split.hip: the
// error-compensated FP16 form; m2l_orbit*.hip: the reflection orbits).
#pragma once

#include "engine.h"

namespace fmmx {

// storage of a multipole slot c in the padded layout read by the M2L B
// operand: four segments of KSP = roundup4(ceil(P2/4)) floats
template <int P>
struct MLayout {
  static constexpr int P2 = P * P, KS = (P2 + 3) / 4, KSP = (KS + 3) / 4 * 4, VS = 4 * KSP;
  static __host__ __device__ constexpr int at(int c) { return (c / KS) * KSP + c % KS; }
};

// Reflection of an M2L offset through the coordinate planes: with reflection
// bits r = (x, y, z), M2L(reflected offset) = T_r M2L(offset) T_r for the
// diagonal +-1 matrix T_r on the real slots: x flips Re by (-1)^m and Im by
// (-1)^(m+1); y flips Im; z flips both by (-1)^(n+m).  Bit c of mask[r] is set
// where T_r has -1.
template <int P>
struct ReflMask {
  static constexpr int W = (P * P + 31) / 32;
  uint32_t mask[8][W];
  constexpr ReflMask() : mask{} {
    for (int r = 0; r < 8; r++) {
      int c = 0;
      for (int im = 0; im < 2; im++)
        for (int n = 0; n < P; n++)
          for (int m = im; m <= n; m++, c++) {
            int neg = 0;
            if (r & 1) neg ^= (m & 1) ^ im;
            if (r & 2) neg ^= im;
            if (r & 4) neg ^= (n + m) & 1;
            if (neg) mask[r][c >> 5] |= 1u << (c & 31);
          }
    }
  }
  __host__ __device__ constexpr bool neg(int r, int c) const { return (mask[r][c >> 5] >> (c & 31)) & 1u; }
};

// Error-compensated FP16 form of the M2L product (v_mfma_f32_16x16x32_f16):
// an FP32 value x is carried as hi = fp16(x) and lo = fp16(x - hi), and
// A B = Ahi Bhi + Alo Bhi + Ahi Blo up to the dropped Alo Blo term (relative
// size 2^-22), with FP32 accumulation.  The three products are one GEMM over
// a K dimension three times as long: lane group g (lanes 16g..16g+15) of an
// MFMA owns the KS input slots g KS .. g KS + KS - 1 and runs them through 8 KH
// k-positions as three segments of SEG = KS rounded up to even:
//   k-position s = seg SEG + u:  A' = (Ahi, Alo, Ahi)[seg],  B' = (hi, hi, lo)[seg]
// at input slot g KS + u (zero for u >= KS, slots >= P2 and seg >= 3).  The
// multipoles of a box are stored per lane group as hi[SEG], lo[SEG], padding
// (GH halfs), so a lane loads its B' words with NB4 16-byte loads and the
// even SEG keeps every pair of k-positions inside one 32-bit word.
// Operators are scaled by 2^sa_e and multipoles by 2^sb_e (powers of two,
// exact) so that their largest magnitude sits just below 2^14: hi stays in
// range and lo above the FP16 subnormals for all but negligible entries.
template <int P>
struct HLayout {
  static constexpr int P2 = P * P, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, SEG = KS + (KS & 1);
  static constexpr int KH = (3 * SEG + 7) / 8;         // k-steps of 32 (8 per lane group)
  static constexpr int GH = (2 * SEG + 7) / 8 * 8;     // halfs per lane group in a stored box
  static constexpr int VSH = 4 * GH;                   // halfs per stored box
  static constexpr int NB4 = GH / 8;                   // 16-byte loads per lane group
  static constexpr int FRH = KH * MT * 64;             // 16-byte operator fragments
  // 32-bit word of a lane's loaded box holding k-positions s, s+1 (s even):
  // hi, hi, lo segments, then the zero padding words, else -1 (constant zero)
  static __host__ __device__ constexpr int word(int s) {
    return s / SEG < 2 ? (s % SEG) / 2
                       : s / SEG == 2 ? SEG / 2 + (s % SEG) / 2 : (SEG + (s - 3 * SEG) / 2 < GH / 2 ? SEG + (s - 3 * SEG) / 2 : -1);
  }
  // input slot of k-position s of lane group g and its segment (-1: none)
  static __host__ __device__ constexpr int slot(int g, int s) {
    return (s / SEG < 3 && s % SEG < KS && g * KS + s % SEG < P2) ? g * KS + s % SEG : -1;
  }
};
// The same split on v_mfma_f32_32x32x16_f16 (two lane groups of 32 lanes,
// 8 k-positions each per step; output tiles of 32 rows x 32 targets): lane
// group g owns the KS = ceil(P2/2) input slots g KS .. g KS + KS - 1.  Stored
// split multipoles: per box two lane groups of GH halfs (hi[SEG], lo[SEG],
// zero padding).
template <int P>
struct WLayout {
  static constexpr int P2 = P * P, MT = (P2 + 31) / 32, KS = (P2 + 1) / 2, SEG = KS + (KS & 1);
  static constexpr int KH = (3 * SEG + 7) / 8;      // k-steps of 16 (8 per lane group)
  static constexpr int GH = (2 * SEG + 7) / 8 * 8;  // halfs per lane group in a stored box
  static constexpr int VSH = 2 * GH;                // halfs per stored box
  static constexpr int NB4 = GH / 8;                // 16-byte loads per lane group
  static constexpr int FRW = KH * MT * 64;          // 16-byte operator fragments
  // word of a lane's loaded box holding k-positions s, s+1 (s even): hi,
  // hi, lo segments, then the zero padding words, else -1 (constant zero)
  static __host__ __device__ constexpr int word(int s) {
    return s / SEG < 2 ? (s % SEG) / 2
                       : s / SEG == 2 ? SEG / 2 + (s % SEG) / 2 : (SEG + (s - 3 * SEG) / 2 < GH / 2 ? SEG + (s - 3 * SEG) / 2 : -1);
  }
};

// largest magnitude of the scaled split operands (2^14)
constexpr int SPLIT_TOP = 14;

struct MSplitLevels;
struct M2LLaunch;

// Reflection orbits of the M2L offsets.  T_r (ReflMask) is diagonal, so the
// real slots fall into 8 classes by their signs under the three reflections:
// class kappa (bits x, y, z) holds the slots with T_r = (-1)^popcount(kappa & r).
// The offsets (+-dx, +-dy, +-dz) that one target sees form an orbit, whose
// sum over the sources s_r at the reflected offsets is
//   sum_r T_r A T_r s_r:  row class c, column class kappa:  A(c, kappa) S_{c ^ kappa},
//   S_psi = sum_r (-1)^popcount(psi & r) s_r   (a Walsh-Hadamard transform),
// one dense product for all of them.  A component of magnitude 0 or 3 appears
// with one sign only (3 with the sign of the target's parity), so an orbit
// doubles the axes in a mask D and the transform runs over those.  The seven
// orbits that double every axis are taken as two halves of either z sign, so
// that no product has more than 4 sources (registers): 63 products per target
// instead of 189, numbered by their mask D (orb_start).
//
// Storage of a class: member i (in slot order) is word i / 4 of lane group
// i % 4.  A step of the product takes one word of every class (an octet: 8
// words per lane, position t = class t); the words that at most four classes
// have beyond the octets form a last step of four words (a quad).
constexpr int NORB = 63, ORB_WPG = 8;
// first product of mask D (D = 7: the end); D = 3 holds its own 7 and the 14
// halves of the fully doubled orbits
constexpr __host__ __device__ int orb_start(int D) { return D <= 3 ? 7 * D : 7 * D + 14; }
constexpr __host__ __device__ int orb_mask(int o) { return o < 21 ? o / 7 : o < 42 ? 3 : o / 7 - 2; }
constexpr int NORBOP = 124;  // distinct operators over the eight parity classes
constexpr __host__ __device__ int orb_class(int n, int m, int im) {
  return ((m ^ im) & 1) | im << 1 | ((n + m) & 1) << 2;
}
template <int P>
struct OLayout {
  static constexpr int P2 = P * P, RW = 16;  // rows of a class's output tile
  int size[8];         // slots of a class
  int16_t slot[8][RW * 2];  // class member -> slot, -1 beyond the class
  int no;              // octet steps
  int quad;            // 1: a quad step follows
  int qc[4];           // classes of the quad step (a class with no word left where fewer than four have one)
  constexpr OLayout() : size{}, slot{}, no(0), quad(0), qc{} {
    for (int k = 0; k < 8; k++)
      for (int i = 0; i < RW * 2; i++) slot[k][i] = -1;
    int c = 0;
    for (int im = 0; im < 2; im++)
      for (int n = 0; n < P; n++)
        for (int m = im; m <= n; m++, c++) {
          const int k = orb_class(n, m, im);
          slot[k][size[k]++] = (int16_t)c;
        }
    // the fewest octets that leave words in at most four classes
    for (no = 0;; no++) {
      int left = 0, more = 0;
      for (int k = 0; k < 8; k++) {
        if (size[k] > 4 * no) left++;
        if (size[k] > 4 * no + 4) more++;
      }
      if (left <= 4 && more == 0) {
        quad = left > 0;
        break;
      }
    }
    int nq = 0;
    for (int k = 0; k < 8 && nq < 4; k++)
      if (size[k] > 4 * no) qc[nq++] = k;
    for (int k = 7; k >= 0 && nq < 4; k--)
      if (size[k] <= 4 * no) qc[nq++] = k;
  }
};
template <int P>
struct OConst {
  static constexpr OLayout<P> O{};
  static constexpr int NO = O.no, QUAD = O.quad, NSTEP = NO + QUAD;
  static constexpr int BS = NO * 32 + QUAD * 16;       // floats of a stored box
  // 16-byte fragments of an operator: an octet's hi and lo apart, a quad's in one
  static constexpr int FRS = 8 * 2 * 64, FRQ = 8 * 64, FRO = NO * FRS + QUAD * FRQ;
  static constexpr int ROWS = 8 * OLayout<P>::RW;      // partial sums per target
};
// The general form (m2l_orbit_gen.hip): row classes of more than 16 slots take
// two 16-row tiles, and classes of more words than the octets hold put up to
// two more words of each into one last octet (positions t, t + 4: words NO,
// NO + 1 of class qc[t]), for Helmholtz (GConst: split expansions of two parts,
// whose operator is [[C, -S], [S, C]] for two real operators C and S) and FP64 (FConst).
template <int P>
struct GLayout {
  OLayout<P> O;
  int no, xtra;          // octets of every class, 1: a last octet of the larger ones
  int qc[4];
  int nt;                // row tiles
  int tcls[16], trow[16];  // class and first row of a tile
  constexpr GLayout() : O{}, no(0), xtra(0), qc{}, nt(0), tcls{}, trow{} {
    for (no = 0;; no++) {
      int left = 0, more = 0;
      for (int k = 0; k < 8; k++) {
        if (O.size[k] > 4 * no) left++;
        if (O.size[k] > 4 * no + 8) more++;
      }
      if (left <= 4 && more == 0) {
        xtra = left > 0;
        break;
      }
    }
    int nq = 0;
    for (int k = 0; k < 8 && nq < 4; k++)
      if (O.size[k] > 4 * no) qc[nq++] = k;
    for (int k = 7; k >= 0 && nq < 4; k--)
      if (O.size[k] <= 4 * no) qc[nq++] = k;
    for (int k = 0; k < 8; k++)
      for (int r = 0; r < O.size[k]; r += 16) {
        tcls[nt] = k;
        trow[nt++] = r;
      }
  }
  // class and member of position t of lane group g at step s (member -1: none)
  constexpr int cls(int s, int t) const { return s == no ? qc[t & 3] : t; }
  constexpr int member(int s, int t, int g) const {
    const int m = s == no ? 4 * (no + (t >> 2)) + g : 4 * s + g;
    return m < O.size[cls(s, t)] ? m : -1;
  }
};
template <int P>
struct GConst {
  static constexpr GLayout<P> L{};
  static constexpr int P2 = P * P, PARTS = 2, NO = L.no, XTRA = L.xtra, NSTEP = NO + XTRA, NT = L.nt;
  static constexpr int PBS = NSTEP * 32, BS = PARTS * PBS;  // floats of a stored part, box
  static constexpr int CH = NT * PARTS * 2 * 64, FRO = NSTEP * CH;  // 16-byte fragments of a step, operator
  static constexpr int ROWS = PARTS * NT * 16;                      // partial sums per target
};
// The FP64 form (m2l_orbit_fp64.hip) in the general layout: k-step ks takes one
// word of a class (4 members), two k-steps share a lane's 16-byte word and
// fragment, and the last octet ends with its last word that any class has.
template <int P>
struct FConst {
  static constexpr GLayout<P> L{};
  static constexpr int NO = L.no, XTRA = L.xtra, NSTEP = NO + XTRA, NT = L.nt;
  static constexpr bool two() {
    for (int k = 0; k < 8; k++)
      if (L.O.size[k] > 4 * NO + 4) return true;
    return false;
  }
  static constexpr int NKX = XTRA ? (two() ? 8 : 4) : 0, NKS = 8 * NO + NKX;  // k-steps of the last octet, of all
  static constexpr int NU = NKS / 2, BS = NU * 8;                   // 64-byte units, doubles of a stored box
  static constexpr int CH = 4 * NT * 64, CHX = NKX / 2 * NT * 64;   // 16-byte fragments of an octet, the last one
  static constexpr int FRO = NO * CH + CHX, ROWS = NT * 16;         // fragments of an operator, partial sums per target
  // step of a k-step and its place in it
  static constexpr __host__ __device__ int step(int ks) { return ks / 8; }
  static constexpr __host__ __device__ int place(int ks) { return ks % 8; }
};
inline bool orbit_f64_supported(int p) { return p >= 6 && p <= P_ALL; }
int launch_m2l_orbit_f64(int p, const MSplitLevels& S, const M2LLaunch& A, int nwg, const int4* orbtab, hipEvent_t e0,
                         hipEvent_t e1, hipStream_t stream);
size_t orbit_f64_box(int p);   // doubles of a stored box
size_t orbit_f64_rows(int p);  // partial sums per target
// fragments of the NORBOP operators from all 316 k-major ones
void orbit_f64_fragments(const double* kmaj, int p, std::vector<double>& out);

// launchers of the Helmholtz form (p = 4, 6, 8, 10, 12)
int launch_m2l_orbit_gen(int p, const M2LLaunch& A, int nwg, const int4* orbtab, hipStream_t stream);
int launch_orbit_gen_order(int p, const MSplitLevels& S, hipStream_t stream);
int launch_orbit_gen_reduce(int p, const M2LLaunch& A, hipStream_t stream);
size_t orbit_gen_box_floats(int p);
size_t orbit_gen_frags(int p);
size_t orbit_gen_rows(int p);
// fragments of one operator (C and S; row-major P2 x P2 blocks of leading dimension
// ld), scaled by 2^sa_e
void orbit_gen_fragments(const double* C, const double* S, int ld, int p, int sa_e, uint4* out);
// the distinct base offsets of the orbits, NORBOP of them
void orbit_op_vector(int i, int* d);

// exponent that scaled multipoles stay below: sums of 4 reach up to FP16's 65,504, and
// the dense FP16 forms' resolution (SPLIT_TOP) is kept
constexpr int ORB_TOP = SPLIT_TOP;
// base offset of product o for a target of parity class cls (bits x, y, z) and
// the operator's index in [0, NORBOP)
void orbit_offset(int o, int cls, int* d);
int orbit_op_index(const int* d);
bool m2l_orbit_supported(int p);
// operator fragments of the orbit kernel from all 316 k-major FP64 operators,
// scaled by 2^sa_e: per operator [octet][row class][hi, lo][lane], then the quad
// step's [row class][lane] with hi and lo in one fragment
void orbit_fragments(const double* kmaj, int p, int sa_e, std::vector<uint4>& out);

// One M2L launch can cover several levels: workgroups [wg0, wg0 + nwg) of
// the grid run level `lev` with that level's tiles, splits and buffers.
// FP16 form: Mh (split multipoles), opH (split operators, fragment order),
// mmax (the level's largest |multipole| as float bits) and sa_e.
struct M2LLev {
  const int* cls_cnt;
  const uint32_t* ord;
  const uint32_t* ikey;
  const int* dense_j;
  const float* M;
  float* L;
  float* part;
  const float* opF;
  const int4* offtab;
  unsigned long long* npairs;
  const uint4* Mh;
  const uint4* opH;
  const unsigned* mmax;
  int lev, nb, nbj, nsplit, init, region, gsh, wg0, nwg, sa_e;
};
struct M2LLaunch {
  M2LLev lv[MAXL + 1];  // ascending wg0
  int nlv;
};

// levels of the multipole split (largest magnitude, then the FP16 pairs):
// boxes [off[k], off[k+1]) of the flattened range belong to level k, the
// last of them a zero box (the split multipoles hold nb + 1 boxes)
struct MSplitLevels {
  const float* M[MAXL + 1];
  uint4* Mh[MAXL + 1];
  unsigned* mmax[MAXL + 1];
  long off[MAXL + 2];
  int nl;
  // independent groups of boxes (Helmholtz): each has its own scale, mmax[k][key >> 3 gs],
  // since its potentials do not see the other groups' magnitudes; ng of them (1: none)
  const uint32_t* key[MAXL + 1];
  int gs[MAXL + 1], ng;
  int wide;  // 1: layout of the 32x32x16 kernel (WLayout), 2: orbit kernel (OLayout, FP32), else HLayout
};

// m2l_split.hip
bool m2l_split_supported(int p);
int launch_msplit(int p, const MSplitLevels& S, hipStream_t stream);
// launch shapes: N-tiles per wave nt (1, 2), waves per workgroup wpg (4, 8),
// db: two operator buffers (8 waves, one N-tile; p with split_db_fits)
int launch_m2l_split(int p, const M2LLaunch& A, int nwg, int nt, int wpg, int db, hipStream_t stream);
bool split_db_fits(int p);
// the 32x32x16 form, all 316 operators: nt 2 (32 targets per wave) with 8
// waves and two LDS buffers or 4 waves and one (two workgroups per CU); nt 4
// (64 targets per wave), 4 waves and two buffers; p with split_wide_fits
int launch_m2l_wide(int p, const M2LLaunch& A, int nwg, int wpg, int nt, hipStream_t stream);
bool split_wide_fits(int p);
// the orbit form: workgroups of ORB_WPG waves of 16 targets; partial sums per split
// and target in row-class order (launch_orbit_reduce puts them into the locals)
int launch_morder(int p, const MSplitLevels& S, hipStream_t stream);
int launch_m2l_orbit(int p, const M2LLaunch& A, int nwg, const int4* orbtab, hipStream_t stream);
int launch_orbit_reduce(int p, const M2LLaunch& A, hipStream_t stream);
void split_fragments_wide(const double* kmaj, int count, int p, int sa_e, std::vector<uint4>& out);
// floats of one stored box of the orbit kernel (0: not built for p)
size_t orbit_box_floats(int p);
// 16-byte fragments of one split operator; halfs of one split box
inline size_t split_frag_count(int p) {
  const int P2 = p * p, MT = (P2 + 15) / 16, KS = (P2 + 3) / 4, SEG = KS + (KS & 1), KH = (3 * SEG + 7) / 8;
  return (size_t)KH * MT * 64;
}
inline size_t split_box_halfs(int p) {
  const int KS = (p * p + 3) / 4, SEG = KS + (KS & 1);
  const int KS2 = (p * p + 1) / 2, SEG2 = KS2 + (KS2 & 1);
  const size_t h = std::max<size_t>((size_t)4 * ((2 * SEG + 7) / 8 * 8), (size_t)2 * ((2 * SEG2 + 7) / 8 * 8));
  return std::max(h, orbit_box_floats(p) * 2);
}
// operator fragments of the split form from k-major FP64 operators (count
// of them, P2 x P2 each, element (row i, column k) at [k P2 + i]), scaled by
// 2^sa_e; sa_e from the largest magnitude of n values
void split_fragments(const double* ops, int count, int p, int sa_e, std::vector<uint4>& out);
int split_scale_exp(const double* ops, size_t n);

}  // namespace fmmx
