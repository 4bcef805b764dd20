// Per-child device routines of the gate-count search.  A lane group of GS = 4^n lanes holds one residual
// matrix, lane le = r * N + c owning entry (r, c); for n = 3 a group is a whole wave64.
#pragma once
#include "dev.h"

namespace chz {

// For n = 3 a lane group is the whole wave, so values shared by a group are wave-uniform: reading them through
// readfirstlane keeps them in scalar registers (fewer vector registers live across the T bound).  Smaller groups
// share a wave with other groups and keep such values per lane.
template <int NQ> __device__ __forceinline__ int wuni(int v) {
  if constexpr (NQ == 3) return __builtin_amdgcn_readfirstlane(v);
  else return v;
}
template <int NQ> __device__ __forceinline__ long long wuni64(long long v) {
  if constexpr (NQ == 3)
    return (long long)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                       (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
  else return v;
}

// value of lane q of the lane group (q uniform across the group)
template <int GS> __device__ __forceinline__ uint32_t gget(uint32_t v, int q) {
  if constexpr (GS == 64) return (uint32_t)__builtin_amdgcn_readlane((int)v, q);
  else return (uint32_t)__shfl((int)v, q, GS);
}
template <int GS> __device__ __forceinline__ uint64_t gget64(uint64_t v, int q) {
  return (uint64_t)gget<GS>((uint32_t)v, q) | ((uint64_t)gget<GS>((uint32_t)(v >> 32), q) << 32);
}

// ST_LAST: alive at its search's last level, so no parent of the next one (tallied as alive)
enum : uint8_t { ST_DEAD = 0, ST_ALIVE = 1, ST_FOUND = 2, ST_W2 = 3, ST_W3 = 4, ST_OVF = 6, ST_LAST = 7 };
constexpr uint32_t INFO_NOBOUND = 1u << 31;    // spec without bounds: every child is kept

// x * w^p for a coefficient vector of int32 values (entries below 2^28 in magnitude: no overflow)
__device__ __forceinline__ int4 zrot(int4 v, int p) {
  const int q = p & 3;
  const int nb = -v.y, nc = -v.z, nd = -v.w;
  // w (a, b, c, d) = (-d, a, b, c)
  int r0 = q == 0 ? v.x : q == 1 ? nd : q == 2 ? nc : nb;
  int r1 = q == 0 ? v.y : q == 1 ? v.x : q == 2 ? nd : nc;
  int r2 = q == 0 ? v.z : q == 1 ? v.y : q == 2 ? v.x : nd;
  int r3 = q == 0 ? v.w : q == 1 ? v.z : q == 2 ? v.y : v.x;
  const int m = (p & 4) ? -1 : 0;   // w^4 = -1
  return make_int4((r0 ^ m) - m, (r1 ^ m) - m, (r2 ^ m) - m, (r3 ^ m) - m);
}
__device__ __forceinline__ uint32_t uabs(int v) { return v < 0 ? 0u - (uint32_t)v : (uint32_t)v; }
__device__ __forceinline__ uint32_t zmag(int4 v) { return uabs(v.x) | uabs(v.y) | uabs(v.z) | uabs(v.w); }

// Child residual entry of lane le: (S g^-1)[r][c] = sum_m S[r][x_m] ginv[m][lc], then the group lowers the
// sqrt2 exponent while every entry is divisible by sqrt2 (src/cheese.cu:146-174, :773-817).  Overflow is
// judged before normalisation, where the reference narrows to int32.  Gates whose entries are all units
// +-w^p (every standard gate) rotate coefficients in int32 while the parent's entries stay below 2^28;
// otherwise the update runs in int64 with the general Z[w] product.  Returns false on overflow.
template <int NQ>
__device__ __forceinline__ bool make_child(const int4 *__restrict__ par, int pk, const DevGate &g, int le, int4 &s,
                                           int &k) {
  constexpr int N = 1 << NQ, GS = N * N;
  const int r = le >> NQ, c = le & (N - 1);
  const int nq = g.nq, L = g.L, mask = g.mask;
  const int q0 = g.q[0], q1 = g.q[1], q2 = g.q[2];
  int lc = (c >> q0) & 1;
  if (nq > 1) lc |= ((c >> q1) & 1) << 1;
  if (nq > 2) lc |= ((c >> q2) & 1) << 2;
  const int base = c & ~mask;
  bool of = false;
  const bool small = gall<GS>(zmag(par[r * N + c]) < (1u << 28));
  if (g.unit && small) {
    int4 acc = make_int4(0, 0, 0, 0);
    for (int m = 0; m < L; m++) {
      const int p = g.ph[m * L + lc];
      if (p < 0) continue;
      int x = base | ((m & 1) << q0);
      if (nq > 1) x |= ((m >> 1) & 1) << q1;
      if (nq > 2) x |= ((m >> 2) & 1) << q2;
      const int4 t = zrot(par[r * N + x], p);
      acc.x += t.x; acc.y += t.y; acc.z += t.z; acc.w += t.w;
    }
    s = acc;
  } else {
    long long a = 0, b = 0, cc = 0, d = 0;
    for (int m = 0; m < L; m++) {
      const int4 gm = g.inv[m * L + lc];
      if (zzero(gm)) continue;
      int x = base | ((m & 1) << q0);
      if (nq > 1) x |= ((m >> 1) & 1) << q1;
      if (nq > 2) x |= ((m >> 2) & 1) << q2;
      const int4 v = par[r * N + x];
      a += (long long)v.x * gm.x - (long long)v.y * gm.w - (long long)v.z * gm.z - (long long)v.w * gm.y;
      b += (long long)v.x * gm.y + (long long)v.y * gm.x - (long long)v.z * gm.w - (long long)v.w * gm.z;
      cc += (long long)v.x * gm.z + (long long)v.y * gm.y + (long long)v.z * gm.x - (long long)v.w * gm.w;
      d += (long long)v.x * gm.w + (long long)v.y * gm.z + (long long)v.z * gm.y + (long long)v.w * gm.x;
    }
    of = a != (int)a || b != (int)b || cc != (int)cc || d != (int)d;
    s = make_int4((int)a, (int)b, (int)cc, (int)d);
  }
  k = pk + g.ik;
  if (gany<GS>(of)) return false;
  while (k > 0 && gall<GS>(zhalf(s))) { s = zdown(s); k--; }
  return true;
}

// Children of unit gates with at most two terms per column and parents below 2^28 (all others: make_child), in two parts:
// the parent entries a lane needs, by its entry descriptor (LevelTabs::sdesc), and the child entry from them.  The
// loads of several children can then be in flight together.  par: the parent's entries in global memory.
struct ChildTerms { int4 a, b; };
template <int NQ> __device__ __forceinline__ ChildTerms child_terms(const int4 *__restrict__ par, uint32_t desc, int le) {
  constexpr int N = 1 << NQ;
  const int4 *row = par + (le >> NQ) * N;
  ChildTerms t;
  t.a = row[desc & 7];
  t.b = desc & 0x1000u ? row[(desc >> 6) & 7] : make_int4(0, 0, 0, 0);
  return t;
}
// false when the parent's entries are too large for the rotations, or the gate is none of these
template <int NQ> __device__ __forceinline__ bool child_of(ChildTerms t, uint32_t desc, int ik, int pk, int4 &s, int &k) {
  constexpr int GS = 1 << (2 * NQ);
  if (!gall<GS>(!(desc & 0x8000u) && (zmag(t.a) | zmag(t.b)) < (1u << 28))) return false;
  s = zrot(t.a, (desc >> 3) & 7);
  if (desc & 0x1000u) {
    const int4 u = zrot(t.b, (desc >> 9) & 7);
    s.x += u.x; s.y += u.y; s.z += u.z; s.w += u.w;
  }
  k = pk + ik;
  while (k > 0 && gall<GS>(zhalf(s))) { s = zdown(s); k--; }
  return true;
}

// 2 if the matrix is monomial with a column permutation that is not affine over GF(2) (src/cheese.cu:321-338);
// b = group ballot of the nonzero entries
template <int NQ> __device__ __forceinline__ int h_struct(uint64_t b) {
  constexpr int N = 1 << NQ;
  if (__popcll(b) != N) return 0;
  uint64_t col0 = 0;
#pragma unroll
  for (int r = 0; r < N; r++) col0 |= 1ull << (r * N);
  int pi[N];
#pragma unroll
  for (int c = 0; c < N; c++) {
    const uint64_t cb = (b >> c) & col0;
    if (__popcll(cb) != 1) return 0;
    pi[c] = (__ffsll((long long)cb) - 1) / N;
  }
#pragma unroll
  for (int j = 0; j < N; j++) {
    int x = pi[0];
#pragma unroll
    for (int i = 0; i < NQ; i++) if ((j >> i) & 1) x ^= pi[1 << i] ^ pi[0];
    if (pi[j] != x) return 2;
  }
  return 0;
}

// entries (r, c) with bit q of r and c different, as a group-local lane mask
template <int NQ> __host__ __device__ constexpr uint64_t offdiag_mask(int q) {
  constexpr int N = 1 << NQ, GS = N * N;
  uint64_t m = 0;
  for (int le = 0; le < GS; le++)
    if ((((le / N) ^ (le % N)) >> q) & 1) m |= 1ull << le;
  return m;
}

// qubits the matrix acts on non-trivially (src/cheese.cu:305-319), as a mask; b = group ballot of the nonzero
// entries.  A nonzero entry off the qubit's diagonal blocks settles that qubit without comparing blocks.
// Only the qubits in `ask` are looked at: a gate leaves the others as trivial or not as they were in the parent.
template <int NQ> __device__ __forceinline__ int support_mask(int4 s, int le, uint64_t b, int ask) {
  constexpr int N = 1 << NQ, GS = N * N;
  const int r = le >> NQ, c = le & (N - 1);
  int m = 0;
#pragma unroll
  for (int q = 0; q < NQ; q++) {
    const int bit = 1 << q;
    if (!(ask & bit)) continue;
    if (b & offdiag_mask<NQ>(q)) { m |= bit; continue; }
    const int4 o = gxor<GS>(s, bit * N + bit);
    const bool viol = !((r | c) & bit) && !zeq(s, o);
    m |= gany<GS>(viol) ? bit : 0;
  }
  return m;
}

__host__ __device__ inline int spread_bits(int v, int mask, int n) {   // bit j of v -> j-th set bit of mask
  int out = 0, j = 0;
  for (int q = 0; q < n; q++)
    if ((mask >> q) & 1) { out |= ((v >> j) & 1) << q; j++; }
  return out;
}

// rank over F_p of the operator-Schmidt matrix across cut A (|A| = sa), R = 4^sa rows, counting up to `stop`
// (src/cheese.cu:270-303).  Lane le holds matrix entry (le / C, le % C).  Full pivoting: any nonzero entry
// of a row not yet used becomes the pivot and its column is cleared from the other unused rows by
// fraction-free updates (each a nonzero multiple of an F_p row combination), so after r steps the rank
// is r plus that of the unused rows; the rank over F_p does not depend on the pivot order.
// Lane le of the matrix across cut A (|A| = sa) holds entry (le >> lgC, le & (C - 1)), C = 2^lgC = 4^(n - sa):
// row (output bits, input bits) on A, column the same on the other qubits.  The residual entry it reads:
template <int NQ> __host__ __device__ inline int cut_source(int le, int A, int sa) {
  constexpr int N = 1 << NQ;
  const int lgC = 2 * (NQ - sa);
  const int mrow = le >> lgC, mcol = le & ((1 << lgC) - 1);
  const int nb = NQ - sa;
  const int ia = mrow & ((1 << sa) - 1), oa = mrow >> sa, ib = mcol & ((1 << nb) - 1), ob = mcol >> nb;
  const int notA = ((1 << NQ) - 1) & ~A;
  const int o = spread_bits(oa, A, NQ) | spread_bits(ob, notA, NQ);
  const int i = spread_bits(ia, A, NQ) | spread_bits(ib, notA, NQ);
  return o * N + i;
}

// src: cut_source of this lane, staged once per kernel; rows and columns are split by shifts (C is a power of 2)
template <int NQ> __device__ __forceinline__ int cut_rank(uint32_t fp, int le, int src, int sa, int stop) {
  constexpr int N = 1 << NQ, GS = N * N;
  (void)N;
  const int lgC = 2 * (NQ - sa), cm = (1 << lgC) - 1;
  const int mrow = le >> lgC, mcol = le & cm;
  uint32_t v = __shfl(fp, src, GS);
  int used = 0, rank = 0;                        // rows already pivots
  while (rank < stop) {
    const bool mine = !((used >> mrow) & 1);
    const uint64_t bb = gballot<GS>(mine && v != 0);
    if (!bb) break;
    if (rank + 1 == stop) return stop;          // the rank reaches the cap: no need to eliminate this pivot
    const int p = __ffsll((long long)bb) - 1;
    const int prow = p >> lgC, pcol = p & cm;
    const uint32_t pv = __shfl(v, p, GS);
    const uint32_t fr = __shfl(v, (mrow << lgC) + pcol, GS);
    const uint32_t pr = __shfl(v, (prow << lgC) + mcol, GS);
    used |= 1 << prow;
    if (mine && mrow != prow) v = mont_mul2(v, pv, fr, pr ? P_MOD - pr : 0u);      // v pv - fr pr
    rank++;
  }
  return rank;
}

// Bound word carried by every frontier node: bits 0-7 its raw T bound (BW_TUNK: not known), bits 8 + 3 i the
// need of cut i (ceil log2 of its clipped rank, at most 2 for n <= 3), bit 30 set when one of its children is
// the goal, bit 31 set when the cut needs are known.  Roots carry BW_TUNK.  A child copies what its gate cannot
// change and computes the rest.
constexpr uint32_t BW_TUNK = 0xffu, BW_CUTS = 1u << 31, BW_GOAL = 1u << 30, BW_NEEDS = 0x1fffff00u;
constexpr int BW_MAXCUTS = 7;
// A survivor's word carries the symmetry of its class key's image (class_key3) in bits 24-27 until the gather, where the
// spec has at most BW_IMAGE_CUTS cuts.
constexpr int BW_IMAGE = 24, BW_IMAGE_CUTS = 5;

// CX/CZ lower bound from the cut ranks and the ILP table (src/cheese.cu:585-597).  Cuts in `keepc` take the
// need packed in `needs` (the parent's: the gate acts on one side of them, so the rank is unchanged); the
// others are ranked here.  On return `needs` holds this matrix's packed needs.
// The cx table is read from the expansion kernel's LDS copy `cxl` when it fits (sp.cxlds): the global table sits
// behind a vector load on every child's dependency chain.
// STD (here and below): the spec is one the expansion's specialised kernel takes (std_spec)
template <bool STD> __device__ __forceinline__ int cx_at(const KSpec &sp, const uint8_t *cxl, int idx) {
  return STD || sp.cxlds ? (int)cxl[idx] : sp.cxtable[idx];
}
template <int NQ, bool STD> __device__ __forceinline__ int n_cuts_of(const KSpec &sp) { return STD ? (NQ == 3 ? 3 : 1) : sp.ncuts; }

// The least a child's cuts can need, from its parent's packed needs: each need drops by at most the gate's per-cut delta
// (operator-Schmidt ranks multiply; 7: by any amount).  low: the needs, packed; idx: their place in the cx table; c2: the
// cut bound there, a lower bound on the child's since the table is non-decreasing in every need.
struct CutLow { uint32_t low; int idx, c2; };
template <int NQ, bool STD>
__device__ __forceinline__ CutLow cut_low(const KSpec &sp, const uint8_t *cxl, uint32_t pneeds, uint32_t cdel) {
  CutLow o{0, 0, 0};
  int mult = 1, mx = 0;
#pragma unroll
  for (int i = 0; i < n_cuts_of<NQ, STD>(sp); i++) {
    const int dl = (int)((cdel >> (3 * i)) & 7u);
    int nd = (int)((pneeds >> (3 * i)) & 7u) - dl;
    nd = dl == 7 || nd < 0 ? 0 : nd;
    o.low |= (uint32_t)nd << (3 * i);
    o.idx += nd * mult;
    mult *= STD ? 3 : sp.rad[i];
    if (nd > mx) mx = nd;
  }
  o.c2 = STD || sp.have_table ? cx_at<STD>(sp, cxl, o.idx) : mx;
  return o;
}

// Bounds known before the cuts of a child: the smallest cut needs its parent leaves (CutLow) and whether they may be
// used, its T bound's lower end, and the other arguments of the bound.  Once the needs found so far and the smallest
// possible others put the child over its budget, the remaining ranks are left out (the value returned is then that lower
// cut bound, and `needs` is not the child's).
struct CutStop { bool on; uint32_t low; int lo, T, h, supp, rem; };

// The need of a cut of one qubit, whose rank is clipped at 3: 0, 1 or 2 for a rank of at most 1, 2 or more.  v: the
// operator-Schmidt matrix, 4 rows of 4^(n - 1) lanes, in F_p.  v pv - fr pr is zero in the pivot's row and column by
// itself, so no row needs to be masked, and two eliminations decide.
template <int NQ> __device__ __forceinline__ int cut_need1(uint32_t v, int le) {
  constexpr int GS = 1 << (2 * NQ), C = GS / 4;
  int need = 0;
#pragma unroll
  for (int step = 0; step < 2; step++) {
    const uint64_t bb = gballot<GS>(v != 0);
    if (!bb) return need;
    need = step;
    const int p = __ffsll((long long)bb) - 1;
    const uint32_t pv = gget<GS>(v, p);
    const uint32_t fr = __shfl(v, (le & ~(C - 1)) | (p & (C - 1)), GS);
    const uint32_t pr = __shfl(v, (p & ~(C - 1)) | (le & (C - 1)), GS);
    v = mont_mul2(v, pv, fr, pr ? P_MOD - pr : 0u);
  }
  return gany<GS>(v != 0) ? 2 : need;
}

// need of cut i of a matrix with the F_p image fp
template <int NQ, bool STD> __device__ __forceinline__ int cut_need(uint32_t fp, int le, const KSpec &sp, const uint8_t *csrc, int i) {
  constexpr int GS = 1 << (2 * NQ);
  if (STD || sp.cut1) return cut_need1<NQ>((uint32_t)__shfl(fp, (int)csrc[i * GS + le], GS), le);
  const int rad = sp.rad[i], sa = sp.cutsize[i];
  const int R = 1 << (2 * sa);
  int stop = R;
  if (rad >= 2 && rad - 2 < 30 && (1 << (rad - 2)) + 1 < stop) stop = (1 << (rad - 2)) + 1;
  const int src = i < CSRC_MAX ? (int)csrc[i * GS + le] : cut_source<NQ>(le, sp.cutmask[i], sa);
  const int rk = cut_rank<NQ>(fp, le, src, sa, stop);
  int need = 0;
  while ((1 << need) < rk) need++;
  return need > rad - 1 ? rad - 1 : need;
}

template <int NQ, bool STD> __device__ __forceinline__ int cx_bound(int4 s, int le, const KSpec &sp, const uint8_t *cxl,
                                                          const uint8_t *csrc, uint32_t keepc, bool small, const CutStop &st,
                                                          uint32_t &needs, uint32_t &ranks) {
  uint32_t fp = 0;
  bool have_fp = false;
  const int nc = n_cuts_of<NQ, STD>(sp);
  int idx = 0, mult = 1, mx = 0, lo = st.lo;
  uint32_t out = 0;
  int todo = nc - __popc(keepc & ((1u << nc) - 1));
#pragma unroll 1
  for (int i = 0; i < nc; i++) {
    int need;
    if ((keepc >> i) & 1) need = (int)((needs >> (3 * i)) & 7u);
    else {
      if (!have_fp) { fp = STD || small ? fp_of_small(s) : fp_of(s); have_fp = true; }
      need = cut_need<NQ, STD>(fp, le, sp, csrc, i);
      ranks++;
      if (st.on && --todo > 0) {
        lo += (need - (int)((st.low >> (3 * i)) & 7u)) * mult;
        const int c = wuni<NQ>(cx_at<STD>(sp, cxl, lo));
        if (st.T > t_budget(st.h, c, st.supp, st.rem) * sp.tdiv) return c;
      }
    }
    if (i < BW_MAXCUTS) out |= (uint32_t)need << (3 * i);
    idx += need * mult;
    mult *= STD || sp.cut1 ? 3 : sp.rad[i];
    if (need > mx) mx = need;
  }
  needs = out;
  return STD || sp.have_table ? wuni<NQ>(cx_at<STD>(sp, cxl, idx)) : mx;
}

// T lower bound: max over Pauli pairs of 2(n+k) - v(X_ab), all X_ab by one 2-D Walsh-Hadamard transform
// per flip pair f = (fa, fb) of Q_f[e] = S[e ^ f] conj(S[e]), arithmetic in Z[w] mod 2^bits(U)
// (src/cheese.cu:397-449).  The minimum valuation over all transforms is read from two OR accumulators:
// O = OR of all coefficients, D = OR of (a ^ c) | (b ^ d); min v = 2 m + [bit m of D clear], m = ctz(O).
template <int NQ, typename U> __device__ __forceinline__ int t_bound(int4 s, int k, int le) {
  constexpr int N = 1 << NQ, GS = N * N;
  const U ya = (U)(long long)s.x, yb = (U)0 - (U)(long long)s.w, yc = (U)0 - (U)(long long)s.z,
          yd = (U)0 - (U)(long long)s.y;
  U O = 0, D = 0;
  for (int f = 0; f < GS; f++) {
    const int4 xs = gxor<GS>(s, f);
    const U xa = (U)(long long)xs.x, xb = (U)(long long)xs.y, xc = (U)(long long)xs.z, xd = (U)(long long)xs.w;
    U qa = U(xa * ya - xb * yd - xc * yc - xd * yb);
    U qb = U(xa * yb + xb * ya - xc * yd - xd * yc);
    U qc = U(xa * yc + xb * yb + xc * ya - xd * yd);
    U qd = U(xa * yd + xb * yc + xc * yb + xd * ya);
#pragma unroll
    for (int h = 1; h < GS; h <<= 1) {
      const U oa = __shfl_xor(qa, h, GS), ob = __shfl_xor(qb, h, GS), oc = __shfl_xor(qc, h, GS),
              od = __shfl_xor(qd, h, GS);
      if (le & h) { qa = U(oa - qa); qb = U(ob - qb); qc = U(oc - qc); qd = U(od - qd); }
      else { qa = U(qa + oa); qb = U(qb + ob); qc = U(qc + oc); qd = U(qd + od); }
    }
    O |= qa | qb | qc | qd;
    D |= (qa ^ qc) | (qb ^ qd);
  }
  O = gor<GS>(O);
  D = gor<GS>(D);
  if (!O) return 0;
  const int m = __ffsll((unsigned long long)O) - 1;
  const int v = 2 * m + (((D >> m) & 1) ? 0 : 1);
  const int need = 2 * (NQ + k) - v;
  return need > 0 ? need : 0;
}

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ u16x2 pk(int lo, int hi) { u16x2 r; r.x = (unsigned short)lo; r.y = (unsigned short)hi; return r; }
__device__ __forceinline__ uint32_t bits(u16x2 v) { return (uint32_t)v.x | ((uint32_t)v.y << 16); }

// Per-entry operands of the packed transform, staged in LDS by the lane owning entry e, 16 bytes each: x[e] =
// (a, b | c, d) of S[e] mod 2^16, and p[e] the four packed multipliers of conj(S[e]) = (a, -d, -c, -b) for the pass at
// hand.  With Q = S[x] conj(S[e]) = (Qa, Qb, Qc, Qd) the transform needs only Qa, Qc and Qb -+ Qd (below), in two passes:
//   (Qa | Qc)           = xa (a | -c)    + xb (b | -d)    + xc (c | a)     + xd (d | b)
//   (Qb - Qd | Qb + Qd) = xa (b-d | -b-d) + xb (a+c | a-c) + xc (b+d | b-d) + xd (c-a | c+a)
constexpr int TS_STRIDE = 256;      // entries per field: one per thread of a block
struct TStage {
  char *lds;                        // a block's p[TS_STRIDE], then its x[TS_STRIDE], aligned to a wave's share
  uint32_t group;                   // byte offset of this group's first entry in either
};

template <int NQ> __device__ __forceinline__ void t_stage_x(TStage st, int4 s, int le) {
  *(uint2 *)(st.lds + 16 * TS_STRIDE + (st.group | (uint32_t)le << 4)) = make_uint2(bits(pk(s.x, s.y)), bits(pk(s.z, s.w)));
}
template <int NQ> __device__ __forceinline__ void t_stage_p(TStage st, int4 s, int le, int pass) {
  const int a = s.x, b = s.y, c = s.z, d = s.w;
  const uint4 p = pass ? make_uint4(bits(pk(b - d, -b - d)), bits(pk(a + c, a - c)), bits(pk(b + d, b - d)), bits(pk(c - a, c + a)))
                       : make_uint4(bits(pk(a, -c)), bits(pk(b, -d)), bits(pk(c, a)), bits(pk(d, b)));
  *(uint4 *)(st.lds + (st.group | (uint32_t)le << 4)) = p;
}

__device__ __forceinline__ u16x2 as16(uint32_t v) { u16x2 r; r.x = (unsigned short)v; r.y = (unsigned short)(v >> 16); return r; }

__device__ __forceinline__ int ctz16(uint32_t v) { return v & 0xffffu ? __ffs((int)(v & 0xffffu)) - 1 : 16; }

// T bound with arithmetic mod 2^16 (exact when n + k <= 16; a value that is 0 mod 2^16 has valuation >= 32 >=
// 2(n+k) and cannot raise the bound).  Q_f[e] = S[e ^ f] conj(S[e]) satisfies Q_f[e ^ f] = conj(Q_f[e]), so for
// f != 0, with j the top bit of f and R = {e : e_j = 0}, the 2-D transform is
//   W_f[z] = A[z] +- conj(A[z]),   A[z] = sum_{e in R} (-1)^{e.z} Q_f[e]   (a transform over the other bits),
// and A + conj A = 2a + (b - d) sqrt2, A - conj A = i (2c + (b + d) sqrt2) for A = (a, b, c, d).  An element
// x + y sqrt2 has valuation min(2 v2(x), 2 v2(y) + 1), so the smallest valuation v over all outputs is the
// minimum of three parts, each read from an OR accumulator:
//   f = 0 (Q_0 = |S|^2 = r + y sqrt2, real; transformed by the whole group, one lane per entry): 2 v2(r),
//       1 + 2 v2(y)
//   pass 1, (b - d | b + d) of every A:  1 + 2 v2, at least 1
//   pass 0, (a | c) of every A:          2 + 2 v2, at least 2
// and the bound is 2(n + k) - v.  Each part only lowers v, so 2(n + k) minus the minimum over the parts computed
// so far is a lower bound on the T bound, exact once no remaining part can go below it.  A pass is the costly
// part (E/2 Z[w] products and a transform per lane); the expansion runs them only for children the lower bound
// leaves undecided, the odd pass first (it sets the minimum far more often).

// The staged T bound: the f = 0 part, then pass 1, then pass 0, each only while the lower bound
// max(Tlo, 2(n + k) - v) stays at most tmax (the largest T bound at which the child is alive) and a remaining part
// could still lower v.  Tlo is a lower bound the caller already has (the parent's bracket, a sibling's value).
// Returns the bound reached; exact tells whether it is the T bound (always so when it is at most tmax).  npass
// counts the passes run.  One function with the pass loop inside keeps the pass's LDS reads interleaved with its
// products; split into separate helpers the compiler issued all 64 reads of a pass at once and spilled.
template <int NQ> __device__ __forceinline__ int t_bound16s(TStage st, int4 s, int k, int le, int Tlo, int tmax,
                                                             uint32_t &npass, bool &exact) {
  constexpr int E = 1 << (2 * NQ), H = E / 2, GS = E;
  const int top = 2 * (NQ + k);
  // f = 0: |S[e]|^2 = r + y sqrt2 with r = a^2 + b^2 + c^2 + d^2, y = ab + bc + cd - da, as a pair mod 2^16
  const u16x2 ab = pk(s.x, s.y), bc = pk(s.y, s.z), cd = pk(s.z, s.w), da = pk(s.w, -s.x);
  u16x2 q0 = ab.xx * ab + bc.xx * bc + cd.xx * cd + da.xx * da;
#pragma unroll
  for (int h = 1; h < GS; h <<= 1) {
    const u16x2 o = as16(NQ == 3 ? wave_xor32(bits(q0), h) : (uint32_t)__shfl_xor((int)bits(q0), h, GS));
    // the lanes with bit h set, as a constant mask: compared per lane, the six factors stayed in registers across the
    // child loop and were spilled
    uint64_t hm = 0;
#pragma unroll
    for (int l = 0; l < 64; l++) hm |= (uint64_t)((l & h) != 0) << l;
    q0 = q0 * as16(__builtin_amdgcn_inverse_ballot_w64(hm) ? 0xffffffffu : 0x00010001u) + o;
  }
  // group ORs are uniform over the group: read through readfirstlane (n = 3) they stay in scalar registers
  const uint32_t acc0 = (uint32_t)wuni<NQ>((int)gor<GS>(bits(q0)));
  const uint32_t accG = acc0 & 0xffffu, accY = acc0 >> 16;
  int v = 2 * ctz16(accG);
  const int vy = 1 + 2 * ctz16(accY);
  v = vy < v ? vy : v;
  int T = top - v > Tlo ? top - v : Tlo;
  exact = v <= 1;
  if (exact || T > tmax) return T;
  __builtin_amdgcn_wave_barrier();
  t_stage_x<NQ>(st, s, le);
  // lane f of the group handles flip pair f (lane 0 repeats f = 1; OR-accumulation is idempotent)
  int f = le == 0 ? 1 : le;
  // keep the per-lane LDS address arithmetic inside the child loop: hoisted, it would cost the kernel occupancy
  asm volatile("" : "+v"(f));
  const int j = 31 - __clz(f);
  // entry e of R number i, as byte offsets: bit b of i is bit b of e below j and bit b + 1 from there on.  In the order
  // of a Gray code one XOR leads from an entry to the next and one from e to e ^ f (two thirds of the instructions that
  // inserting the zero bit takes)
  uint32_t vb[2 * NQ - 1];
#pragma unroll
  for (int b = 0; b < 2 * NQ - 1; b++) vb[b] = (b >= j ? 32u : 16u) << b;
  const uint32_t fo = (uint32_t)f << 4;
#pragma unroll 1
  for (int pass = 1; pass >= 0; pass--) {
    __builtin_amdgcn_wave_barrier();
    t_stage_p<NQ>(st, s, le, pass);
    __builtin_amdgcn_wave_barrier();
    // the addresses below depend on a value the compiler cannot see through, so they are formed per pass
    // instead of being hoisted out of the pass loop (64 more live registers)
    uint32_t at = st.group;
    asm volatile("" : "+v"(at));
    u16x2 q[H];
#pragma unroll
    for (int t = 0; t < H; t++) {
      if (t) at ^= vb[t & 1 ? 0 : t & 2 ? 1 : t & 4 ? 2 : t & 8 ? 3 : 4];
      const uint2 xv = *(const uint2 *)(st.lds + 16 * TS_STRIDE + (at ^ fo));
      const uint4 m = *(const uint4 *)(st.lds + at);
      const u16x2 x01 = as16(xv.x), x23 = as16(xv.y);
      q[t ^ (t >> 1)] = x01.xx * as16(m.x) + x01.yy * as16(m.y) + x23.xx * as16(m.z) + x23.yy * as16(m.w);
    }
#pragma unroll
    for (int h = 1; h < H / 2; h <<= 1)
#pragma unroll
      for (int i = 0; i < H; i++)
        if (!(i & h)) {
          const u16x2 u = q[i], w = q[i | h];
          q[i] = u + w;
          q[i | h] = u - w;
        }
    // The last step's sums and differences are wanted for the lowest bit set in any of them: where v2(u) and v2(w)
    // differ it is the lower one, which is the lowest bit of u ^ w; where they agree exactly one of u + w, u - w has
    // valuation v2(u) + 1, the lowest bit of 2 (u & w), and u ^ w has none below it
    uint32_t ox = 0, oa = 0;
#pragma unroll
    for (int i = 0; i < H / 2; i++) {
      const uint32_t u = bits(q[i]), w = bits(q[i | H / 2]);
      ox |= u ^ w;
      oa |= u & w;
    }
    const uint32_t o = ox | (oa << 1 & 0xfffefffeu);
    const uint32_t acc = (uint32_t)wuni<NQ>((int)gor<GS>((o & 0xffffu) | (o >> 16)));
    npass++;
    const int vp = (pass ? 1 : 2) + 2 * ctz16(acc);    // pass 1: 1 + 2 v2 of (b - d | b + d); pass 0: 2 + 2 v2 of (a | c)
    v = vp < v ? vp : v;
    T = top - v > Tlo ? top - v : Tlo;
    exact = pass == 0 || v <= 2;
    if (exact || T > tmax) break;
  }
  __builtin_amdgcn_wave_barrier();
  return T;
}

template <int NQ> __device__ __forceinline__ int t_bound_any(int4 s, int k, int le) {
  return 2 * (NQ + k) <= 64 ? t_bound<NQ, uint32_t>(s, k, le) : t_bound<NQ, unsigned long long>(s, k, le);
}

// 32-bit hash of one entry's four coefficients and of its conjugate's: linear forms with 24-bit products (full rate; a
// 32-bit product runs at a quarter of it), folded once.  Entries that collide differ by a vector of the forms' lattice,
// whose shortest ones have coefficients of some 2^8; the summands below are not linear in them.  Coefficients of more
// than 24 bits enter by their low 24.
__device__ __forceinline__ uint32_t entry_hash32(int4 v) {
  const uint32_t h = (uint32_t)(__mul24(v.x, 0x5e3779) + __mul24(v.y, 0x3ebca7) + __mul24(v.z, 0x72b2ae) + __mul24(v.w, 0x27d4eb));
  return h ^ (h >> 15);
}
__device__ __forceinline__ uint32_t entry_hash32_conj(int4 v) {
  const uint32_t h = (uint32_t)(__mul24(v.x, 0x5e3779) + __mul24(v.w, -0x3ebca7) + __mul24(v.z, -0x72b2ae) + __mul24(v.y, -0x27d4eb));
  return h ^ (h >> 15);
}
// The 64-bit summand of an entry hash at position pos (1..64): a square of the two mixed, one product at a quarter of
// the rate where two mixes took two.  Its halves are summed apart.
__device__ __forceinline__ uint64_t slot64(uint32_t h, uint32_t pos) {
  const uint32_t x = h ^ __umul24(pos, 0x9e3779u);
  return (uint64_t)x * (x ^ 0x5bd1e995u);
}

// class key: the smallest over the symmetry group of an entry-sum hash of sigma(S); equal classes give
// equal keys, and equality of keys is always confirmed exactly (src/cheese.cu:224-241)
template <int NQ> __device__ __forceinline__ uint64_t class_key(int4 s, int k, int le, const KSpec &sp) {
  constexpr int N = 1 << NQ, GS = N * N;
  const int r = le >> NQ, c = le & (N - 1);
  const uint32_t hv = entry_hash32(s), hc = entry_hash32_conj(s);
  uint64_t best = ~0ull;
  for (int y = 0; y < sp.nsym; y++) {
    const uint8_t *pm = sp.symperm + y * N;
    const uint32_t pos = (uint32_t)(pm[r] * N + pm[c]) + 1;
    const uint64_t h = slot64(sp.symconj[y] ? hc : hv, pos);
    const uint64_t key = mix64(((uint64_t)gsum<GS>((uint32_t)(h >> 32)) << 32 | gsum<GS>((uint32_t)h)) ^ ((uint64_t)(k + 1) * 0xc2b2ae3d27d4eb4full));
    best = key < best ? key : best;
  }
  return best;
}

// class_key for n = 3 (one matrix per wave64, whole wave active, at most 16 symmetries).  The group permutes qubits and
// may conjugate, so most of its elements are ruled out before any image is hashed: sums over the entries that do not
// depend on their places tell S from its conjugate, and for each qubit a sum over the entries off the qubit's diagonal
// moves with the qubit.  Only the elements that bring the smaller of the two conjugates and the smallest order of the
// qubits' sums are hashed; equal classes have the same images under these, so the smallest of their hashes is the same.
// Hashing all twelve images of a 3-qubit default set took 410 vector instructions a key and a third of the expansion's
// quarter-rate products; two or three sums and usually one image take about 130.
//   spos[y * 64 + le]: position of entry le under symmetry y; cjm bit y: symmetry y conjugates; adm[order]: the
//   symmetries that bring the qubits' sums into the smallest order, among those that conjugate and among the others,
//   with `order` the number of smaller sums of each qubit in two bits (KeyTab)
// image: the symmetry whose image has the smallest hash; matrices of one class have that image in common, so the dedupe
// compares two of them by it.
struct KeyTab { uint16_t adm[64]; };
__host__ __device__ inline int key_order(uint32_t a, uint32_t b, uint32_t c) {
  return ((b < a) + (c < a)) | ((a < b) + (c < b)) << 2 | ((a < c) + (b < c)) << 4;
}
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  return wave_total32(v, [](uint32_t a, uint32_t b) { return a + b; });
}
__device__ __forceinline__ uint64_t class_key3(int4 s, int k, int lane, const uint8_t *spos, const uint16_t *adm, uint32_t cjm,
                                               int &image) {
  const uint32_t hv = entry_hash32(s), hc = entry_hash32_conj(s);
  const int off = (lane >> 3) ^ (lane & 7);            // bit q: an entry off qubit q's diagonal
  // 64 shares of 10 bits sum within 16 bits: two sums to a word
  auto order = [&](uint32_t h) -> uint32_t {
    const uint32_t x = h & 0x3ffu;
    const uint32_t s01 = wave_sum((off & 1 ? x : 0u) | (off & 2 ? x << 16 : 0u)), s2 = wave_sum(off & 4 ? x : 0u);
    return adm[key_order(s01 & 0xffffu, s01 >> 16, s2)];
  };
  uint32_t m;
  if (!cjm) m = order(hv);
  else {
    const uint32_t t = wave_sum(hv >> 22 | (hc >> 22) << 16), tv = t & 0xffffu, tc = t >> 16;
    m = 0;
    if (tv <= tc) m |= order(hv) & ~cjm;
    if (tv >= tc) m |= order(hc) & cjm;
  }
  m = (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
  uint64_t best = ~0ull;
  while (m) {
    const int y = __ffs((int)m) - 1;
    m &= m - 1;
    const uint64_t x = slot64((cjm >> y) & 1 ? hc : hv, (uint32_t)spos[y * 64 + lane] + 1);
    const uint64_t key = (uint64_t)wave_sum((uint32_t)(x >> 32)) << 32 | wave_sum((uint32_t)x);
    if (key < best || best == ~0ull) { best = key; image = y; }
  }
  return mix64(best ^ ((uint64_t)(k + 1) * 0xc2b2ae3d27d4eb4full));
}

// exact: B = sigma(A) for some group element (src/cheese.cu:242-255)
// the same test with the group's entry maps staged in LDS: spos[y * E + e] is the entry of b that lands on entry e
// under group element y, bit y of cjm its conjugation flag
template <int NQ> __device__ __forceinline__ bool same_class_lds(int4 a, int ka, int4 b, int kb, int le,
                                                                const uint8_t *spos, uint32_t cjm, int nsym) {
  constexpr int N = 1 << NQ, GS = N * N;
  if (ka != kb) return false;
  const int4 ac = zconj(a);
  for (int y = 0; y < nsym; y++) {
    const int4 bv = gshfl<GS>(b, spos[y * GS + le]);
    const int4 av = (cjm >> y) & 1 ? ac : a;
    if (gall<GS>(zeq(av, bv))) return true;
  }
  return false;
}

// the same test of b against the image of a representative held in LDS (rep: sigma_y(A) for some group element y, E
// entries): b is of A's class exactly when some group element takes it to that image.  `first` is tried before the
// others: the symmetry of b's own smallest image, which is nearly always the one
template <int NQ> __device__ __forceinline__ bool same_class_image(int4 b, int kb, const int4 *rep, int krep, int first, int le,
                                                                  const uint8_t *spos, uint32_t cjm, int nsym) {
  constexpr int GS = (1 << NQ) * (1 << NQ);
  if (kb != krep) return false;
  const int4 bc = zconj(b);
  auto hit = [&](int y) { return gall<GS>(zeq((cjm >> y) & 1 ? bc : b, rep[spos[y * GS + le]])); };
  if (hit(first)) return true;
  for (int y = 0; y < nsym; y++)
    if (y != first && hit(y)) return true;
  return false;
}

template <int NQ> __device__ __forceinline__ bool same_class(int4 a, int ka, int4 b, int kb, int le, const KSpec &sp) {
  constexpr int N = 1 << NQ, GS = N * N;
  if (ka != kb) return false;
  const int r = le >> NQ, c = le & (N - 1);
  for (int y = 0; y < sp.nsym; y++) {
    const uint8_t *pm = sp.symperm + y * N;
    const int4 bv = gshfl<GS>(b, pm[r] * N + pm[c]);
    const int4 av = sp.symconj[y] ? zconj(a) : a;
    if (gall<GS>(zeq(av, bv))) return true;
  }
  return false;
}

}  // namespace chz
