// Gate-count search on one MI355X: per-level expansion, T bound, ordered compaction, LDS-staged LSD radix
// sort, segmented exact dedupe and frontier gather, all hand-written HIP kernels for gfx950, driven by the
// C-ABI in include/cheese_hip.h.  Reference behaviour: src/cheese.cu:1249-1377 (levels), :1762-1848 (run).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <deque>
#include <map>
#include <memory>
#include <string>
#include <vector>

#include "../../include/cheese_hip.h"
#include "host.h"
#include "primitives.h"
#include "search_kernels.h"
#include "spec.h"

static int verify_hs(const chz::HostSpec &hs, const int *circuit, int len);

namespace chz {

// ------------------------------------------------------------------------------------------------------
// counters of one level (device): indices into a u64 array
// C_EVAL children past the windows, C_PRE those of them settled from the parent's bounds (the others' residuals are
// formed), C_CHEAP through the structural bounds, C_CUTS cut ranks computed,
// C_NEEDT T-bound evaluations (their f = 0 parts), C_KEYS class keys, C_TPASS flip-pair passes of the T bound: the
// stage counts of the expansion's work model
// C_M, C_NCC: the level's parents and children, written by the host with the level's control upload (read by the
// kernels of a captured level step, whose launches are sized for a capacity)
enum { C_W2 = 0, C_W3, C_DEAD, C_FOUND, C_ALIVE, C_OVF, C_NEEDT, C_FIRST, C_REPOVF, C_KEPT, C_EVAL, C_SURV,
       C_CHEAP, C_CUTS, C_KEYS, C_TPASS, C_PRE, C_M, C_NCC, C_N };
// per-instance counters of one level (a batch carries several searches that share the spec's gate set)
enum { IC_W2 = 0, IC_W3, IC_DEAD, IC_FOUND, IC_ALIVE, IC_OVF, IC_FIRST, IC_N };

// The expansion's blocks add up their waves' counts in LDS and add them to the counters in the stripe of their block
// number; the host sums the stripes.  With every wave adding its 13 counts (2 qubits: 31) to one set of counters, the
// additions to one cache line, 2 to 4 ns each whatever the kernel did meanwhile, set the time of levels of up to some
// ten thousand parents: a 2-qubit level of 28 thousand parents took 855 us, its next one without counts 58.  Expansion
// of eight 2-qubit searches 12.9 -> 2.2 ms, of the budget-9 Toffoli proof 0.35 -> 0.17 ms.
enum { SG_EVAL = 0, SG_PRE, SG_NEEDT, SG_CHEAP, SG_CUTS, SG_KEYS, SG_TPASS, SG_N = 8 };
constexpr int NSTRIPE = 16;
static int slot_stripes(int ns) { return std::max(1, std::min(NSTRIPE, 256 / ns)); }    // of the per-slot counters
// words of the counters: [C_N | stage stripes | slot stripes | slot bounds]
static size_t bounds_at(int ns) { return (size_t)C_N + (size_t)NSTRIPE * SG_N + (size_t)slot_stripes(ns) * ns * IC_N; }
static size_t counter_words(int ns) { return bounds_at(ns) + 2 * (size_t)ns; }

struct ExpandArgs {
  const int4 *res;          // parents' residuals, E entries each
  const int *pk;            // parents' sqrt2 exponents
  const uint8_t *g1, *g2;   // parents' last / second-to-last gates (255: none)
  long long off;            // first parent of the chunk (index in the level)
  uint8_t *status;          // per child of the chunk
  uint64_t *keys;           // class keys of kept children
  uint32_t *info;           // bound words of kept children
  const uint32_t *pb;       // parents' bound words
  const uint64_t *tm;       // parents' T columns (k_tcols; n = 3, specialised kernel)
  unsigned long long *stage;  // NSTRIPE stripes of the stage counts (SG_N each)
  const uint32_t *pinst;    // instance slot of every parent of the level (null: one instance, slot 0)
  const int *rem;           // per slot: gate budget left after this level's gate (depth - t)
  const uint8_t *keepi;     // per slot: this level's survivors become parents (t < depth)
  unsigned long long *icnt; // per slot: IC_N counters, in nstr stripes istride apart
  int nstr, istride;
  int gsplit;               // a parent's candidates are split among this many lane groups (small levels)
  const unsigned long long *npd;   // parents read on the device (captured step; gsplit then from tw), or null
  int tw;                   // candidate-split threshold in waves (with npd)
  int psplit;               // lane groups per parent up to which children are settled from the parent's bounds (pre_split)
  const uint32_t *gflag;    // per slot: some parent of the level has a goal child (null: not tracked)
};

// One level's children, fused (src/cheese.cu:662-720, :959-1021): a lane group per parent holds the parent's
// residual in LDS and walks all G candidates: windows, child residual, overflow, goal, cheap bounds, T bound
// (mod 2^16, one lane per flip pair, when n + k <= 16; else mod 2^32 / 2^64, one lane per entry) and the
// class key of a kept child.  Writes the status byte (and key) of every child of the chunk.
constexpr int MAXG = 64;
constexpr int PRE_SPLIT = 4;    // lane groups per parent up to which children are settled from the parent's bounds

// The expansion kernel's LDS tables, built once per context on the host (build_level_tabs) and copied into LDS by
// every block with coalesced 16-byte loads; built inside the kernel they cost each block scattered global loads,
// which small levels (one parent per wave) cannot amortise.
struct LevelTabs {
  // per candidate and entry (g * 64 + e), the child entry's terms for unit gates with at most two per column (Parent):
  // bits 0-5 ring word of the first term in its row, 6 its sign, 7-12 and 13 the second, 14 two terms
  uint16_t term[MAXG * 64];
  // per candidate: x: bits 0-7 tdel (at most 255), 8-10 qubits, 11-15 the most the sqrt2 exponent can fall (0 for a
  // permutation of unit entries, which leaves divisibility by sqrt2 as it is, else the gate's own exponent), 16 an H
  // (the exponent is read off the parent exactly), 24-31 1 + the T-bound class; y: DevGate::cdel; z: DevGate::ik;
  // w: bit 0 the terms above form its children, 1 a permutation of unit entries, 8-23 DevGate::cutloc
  uint4 head[MAXG];
  uint64_t keep_cols[MAXG];        // n = 3: the parent's columns that a child keeps as one of its own (form_columns)
  KeyTab kt;                       // n = 3: the class key's choice of symmetries
  uint8_t spos[16 * 64];           // n = 3: position of entry e under symmetry y (y * 64 + e)
  uint8_t scx[CXL_MAX];            // the cx table when it fits (KSpec::cxlds)
  uint8_t scsrc[CSRC_MAX * 64];    // cut i's operator-Schmidt matrix: entry source of lane le (i * GS + le)
};
// the table in device memory: the part above, then what the dedupe and the gather copy
// sdesc: bits 0-2 source column x0, 3-5 power p0 of w, 6-8 x1, 9-11 p1, bit 12 two terms; bit 15: use the table loop
struct SpecTabs {
  LevelTabs level;
  uint16_t sdesc[MAXG * 64];
  uint8_t col_src[MAXG * 64];      // n = 3: gate_columns' src (255: none; form_columns)
};
static_assert(sizeof(LevelTabs) % 16 == 0, "LevelTabs is copied as uint4");

// A parent's residual in LDS: each entry a + b w + c w^2 + d w^3 as the seven words -b, -c, -d, a, b, c, d, of which the
// four from word 3 - p on are the entry times w^p (w^4 = -1), for p up to 3; a sign gives the other powers.  A child's
// term is then two two-word reads, where rotating a coefficient vector in registers took some 30 instructions.  The odd
// stride keeps the lanes of a row on different banks.
constexpr int RING = 7;
// the identity's nonzero entries
template <int NQ> __host__ __device__ constexpr uint64_t ident_mask() {
  uint64_t m = 0;
  for (int i = 0; i < 1 << NQ; i++) m |= 1ull << (i * (1 << NQ) + i);
  return m;
}
template <int NQ> struct Parent {
  int *e;                          // the group's entries
  int c;                           // this lane's column
  const int *row;                  // this lane's row of entries
  __device__ __forceinline__ void put(int le, int4 v) const {
    int *w = e + le * RING;
    w[0] = (int)(0u - (uint32_t)v.y); w[1] = (int)(0u - (uint32_t)v.z); w[2] = (int)(0u - (uint32_t)v.w);
    w[3] = v.x; w[4] = v.y; w[5] = v.z; w[6] = v.w;
  }
  __device__ __forceinline__ int4 entry(int i) const {
    const int *w = e + i * RING + 3;
    return make_int4(w[0], w[1], w[2], w[3]);
  }
  // the entry and turn at `word` of this lane's row
  __device__ __forceinline__ int4 turned(uint32_t word) const {
    const int *w = row + word;
    return make_int4(w[0], w[1], w[2], w[3]);
  }
};

// the expansion's class key outside it: the tables read from their global copy
template <int NQ> __device__ __forceinline__ uint64_t node_key(int4 s, int k, int le, const KSpec &sp) {
  if constexpr (NQ == 3) {
    const LevelTabs *t = &((const SpecTabs *)sp.ktab)->level;
    int image = 0;
    return class_key3(s, k, le, t->spos, t->kt.adm, sp.cjm, image);
  } else {
    return class_key<NQ>(s, k, le, sp);
  }
}

// STD: the kernel of the specs and levels that std_level accepts (bounds on, the identity as the goal, one table of
// one-qubit cuts in LDS, unit gates of at most two terms a column, coefficients and exponents that no child of the level
// can take out of the fast forms).  It leaves out every other form; carried along, they cost the child loop registers,
// spilled scalars and branches (budget-14 proof 104.4 ms without this kernel, 86.4 with it).
template <int NQ, int WPE, bool STD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void k_level(KSpec sp, ExpandArgs a,
                                                                                         long long np) {
  constexpr int N = 1 << NQ, E = N * N, GS = E, CPW = 64 / GS;
  __shared__ __align__(1024) uint4 stage[2 * TS_STRIDE];
  __shared__ int spar[256 * RING];             // each group's parent residual (Parent)
  __shared__ __align__(16) LevelTabs tb;
  for (int i = threadIdx.x; i < (int)(sizeof(LevelTabs) / 16); i += blockDim.x) ((uint4 *)&tb)[i] = sp.ktab[i];
  const uint8_t *const spos = tb.spos, *const scx = tb.scx, *const scsrc = tb.scsrc;
  const uint32_t cjm = NQ == 3 ? sp.cjm : 0u;
  __syncthreads();
  const int lane = threadIdx.x & 63, le = lane & (GS - 1), slot = lane / GS;
  const int r = le >> NQ, c = le & (N - 1);
  const TStage st{(char *)stage, (threadIdx.x & ~(GS - 1)) << 4};
  const Parent<NQ> P{spar + (threadIdx.x & ~(GS - 1)) * RING, c, spar + ((threadIdx.x & ~(GS - 1)) + r * N) * RING};
  const long long wave = wave_index();
  const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
  const int G = sp.G;
  const bool lite = !STD && sp.lite, bounds = STD || sp.standard || sp.lite;
  // per-instance status tallies: one LDS counter per status value and group, bumped by the group's leader lane
  // and flushed when the group's instance changes (32-bit: one wave's share of a launch is far below 2^32
  // children).  Held in registers they cost two vector or scalar instructions per tally and child, and the
  // scalar registers they take push others into spill lanes.
  __shared__ uint32_t stally[256 / GS][8];
  uint32_t *const tl = stally[threadIdx.x / GS];
  for (int i = le; i < 8; i += GS) tl[i] = 0;
  __builtin_amdgcn_wave_barrier();
  uint32_t n_eval = 0, n_pre = 0, n_t = 0, n_cheap = 0, n_cuts = 0, n_keys = 0, n_tp = 0;
  int cur = -1;
  unsigned long long *const icnt = a.icnt + (size_t)(blockIdx.x & (unsigned)(a.nstr - 1)) * a.istride;
  // the counter of a status value
  auto slot_of = [](int st) {
    return st == ST_W2 ? IC_W2 : st == ST_W3 ? IC_W3 : st == ST_DEAD ? IC_DEAD : st == ST_FOUND ? IC_FOUND : st == ST_OVF ? IC_OVF : IC_ALIVE;
  };
  auto flush = [&]() {
    __builtin_amdgcn_wave_barrier();
    if (le == 0 && cur >= 0)
      for (int i = 0; i <= ST_OVF; i++)
        if (const uint32_t v = tl[i]) atomicAdd(&icnt[(size_t)cur * IC_N + slot_of(i)], (unsigned long long)v);
    __builtin_amdgcn_wave_barrier();
    for (int i = le; i < 8; i += GS) tl[i] = 0;
    __builtin_amdgcn_wave_barrier();
  };
  int gsplit = a.gsplit;
  if (a.npd) {
    np = (long long)*a.npd;
    const long long gs = np ? ((long long)a.tw * CPW + np - 1) / np : 1;
    gsplit = (int)(gs < 1 ? 1 : gs > G ? G : gs);
  }
  const long long nitems = np * gsplit;
  const int cs = (G + gsplit - 1) / gsplit;
  for (long long base = wave * CPW; base < nitems; base += nwaves * CPW) {
    const long long item = base + slot;
    if (item >= nitems) continue;
    // readfirstlane keeps the parent and the candidate range (the child loop's bounds) scalar for n = 3; the 64-bit
    // division, some 150 instructions, is only for split parents
    const long long pl = wuni64<NQ>(gsplit == 1 ? item : item / gsplit);
    const int gbeg = wuni<NQ>((int)(item - pl * gsplit) * cs), gend = gbeg + cs < G ? gbeg + cs : G;
    const long long pi = a.off + pl;
    const int inst = wuni<NQ>(a.pinst ? (int)a.pinst[pi] : 0);
    if (inst != cur) { flush(); cur = inst; }
    const int rem = wuni<NQ>(a.rem[inst]);
    const bool keep = wuni<NQ>((int)a.keepi[inst]) != 0;
    const int4 S = a.res[pi * E + le];
    const int pk = wuni<NQ>(a.pk[pi]), g1 = wuni<NQ>((int)a.g1[pi]), g2 = wuni<NQ>((int)a.g2[pi]);
    const uint32_t pbw = (uint32_t)wuni<NQ>((int)a.pb[pi]);
    const uint64_t tcols = STD && NQ == 3 ? (uint64_t)wuni64<NQ>((long long)a.tm[pi]) : 0ull;
    const uint32_t mag = STD ? 0u : zmag(S);
    const bool small = STD || gall<GS>(mag < (1u << 28));
    // A search whose circuit is found at this level ends with it: its parents without a goal child (no
    // BW_GOAL) are passed over once their coefficients rule out an overflowing child.  Goal children come only
    // from BW_GOAL parents, so the level's found count, first circuit and overflow test are unchanged.
    if (a.gflag && !(pbw & BW_GOAL) && wuni<NQ>((int)a.gflag[inst]) != 0 && (STD || gall<GS>(mag <= sp.maglim))) {
      for (int g = gbeg + le; g < gend; g += GS) a.status[pl * G + g] = ST_DEAD;
      continue;
    }
    __builtin_amdgcn_wave_barrier();
    P.put(le, S);
    __builtin_amdgcn_wave_barrier();
    // a child's cut needs can be bounded from its parent's
    const bool cutlow = !lite && (STD || sp.cx_mono) && (pbw & BW_CUTS);
    const uint32_t pneeds = (pbw & BW_NEEDS) >> 8;
    // T bounds of this parent's children per T-bound class: tc_ok bit set when one is known, tc_ex when it is the
    // exact bound, else it is a lower bound (a transform stopped once the child was dead)
    uint64_t tc_val = 0;
    uint32_t tc_ok = 0, tc_ex = 0;
    // Bounds from the parent alone, one candidate per lane: the child's sqrt2 exponent is at least the parent's less
    // what the gate can take, its T bound and cut needs are bracketed as below, and a qubit the gate leaves alone
    // stays as non-trivial as it is in the parent.  The bound combination grows with each of these, so a child that
    // the lower ends put over its budget is dead, and its residual is not formed: on the Toffoli budget-12 proof 2.61
    // of 5.71 million children past the windows still form one (3.12 without the T siblings below).  Only where no child
    // can overflow (which would be reported) and the goal's own bounds are 0 (a goal child is never over its budget).
    // On the budget-14 proof the expansion takes 111 ms instead of 139.  Where a parent's candidates are split over
    // many lane groups each of them would repeat this, which took small levels 5 % longer: PRE_SPLIT.  A parent whose
    // entries sqrt2 divides has children of lower exponents yet; only a root can be one, since a target keeps its exponent
    // as written, and the level of such a root forms every residual (pre_split).
    const bool pre = gsplit <= a.psplit && (STD || (sp.pre && gall<GS>(mag <= sp.maglim)));
    const bool tparent = (pbw & BW_TUNK) != BW_TUNK;
    // H on qubit q pairs the columns c and c ^ 2^q as their sum and difference over sqrt2: the exponent rises by one,
    // less one if sqrt2 divides every sum (the parities of a + c and b + d agree in each pair), less another if 2 does
    // (every coefficient's parity agrees); it falls by no more than one
    int he = 0;                                  // bits q, 4 + q: the first, the second holds for qubit q
    if (pre) {
      // per lane the parities of a, b, c, d (bits 2-5) and of a + c, b + d (bits 0-1), compared with the paired column's: 50
      // scalar instructions a parent fewer than by masks of ballots
      const uint32_t par = (S.x & 1u) | (S.y & 1u) << 1 | (S.z & 1u) << 2 | (S.w & 1u) << 3;
      const uint32_t w = par << 2 | ((par ^ par >> 2) & 3u);
#pragma unroll
      for (int q = 0; q < NQ; q++) {
        const uint32_t d = w ^ (NQ == 3 ? wave_xor32(w, 1 << q) : (uint32_t)__shfl_xor((int)w, 1 << q, GS));
        if (!gany<GS>(d & 3u)) he |= 1 << q;
        if (!gany<GS>(d & 0x3cu)) he |= 16 << q;
      }
    }
    const int pq = !lite ? support_mask<NQ>(S, le, gballot<GS>(!zzero(S)), N - 1) : 0;
    uint64_t w2m = 0, w3m = 0, dm = 0;
    int lim = 1 << 30, tcl = -1;                 // n = 3: candidate `lane`'s largest T bound by these bounds; its T class
    CutLow cl{0, 0, 0};                          // n = 3: candidate `lane`'s least cut needs
    int tlo = 0;                                 // and least T bound
    // window cuts of every candidate of this parent, one candidate per lane, as two bit masks: the candidate
    // loop then tests bits instead of waiting on a table load per child
    for (int b0 = 0; b0 < G; b0 += GS) {
      const int g = b0 + le;
      bool c2 = false, c3 = false, dead = false;
      if (g < G && g1 != 255) {
        c2 = sp.bad2[g1 * G + g] != 0;
        if (g2 != 255) {
          const uint32_t tri = ((uint32_t)g2 * G + g1) * G + g;
          c3 = ((sp.bad3[tri >> 5] >> (tri & 31)) & 1) != 0;
        }
      }
      if ((pre || (NQ == 3 && cutlow)) && g < G) {
        const uint4 hd = tb.head[g];
        const CutLow lo = cutlow ? cut_low<NQ, STD>(sp, scx, pneeds, hd.y) : CutLow{0, 0, 0};
        const int td = (int)(hd.x & 255u), Tp = (int)(pbw & BW_TUNK);
        // The T bound is the largest exponent of the columns of the residual's Pauli transfer matrix.  A column that the
        // gate leaves alone (a T on qubit q: those without X on q) and that attains the parent's bound is the child's
        // too, so the bound cannot fall: 25.9 of 33.7 million T bounds of the budget-14 proof were evaluated to find that
        // it had not
        int T = tparent && td != 255 && Tp > td ? Tp - td : 0;
        if constexpr (NQ == 3) {
          cl = lo;
          if (STD && tparent && (tcols & tb.keep_cols[g])) T = Tp;
          tlo = T;
        }
        if (pre) {
          const uint32_t w = hd.x;
          const int gm = (int)((w >> 8) & 7u), hq = he >> (__ffs(gm) - 1);
          const int kd = (w >> 16) & 1u ? pk + 1 - (hq & 1) - ((hq >> 4) & 1) : pk - (int)((w >> 11) & 31u), h = kd > 0 ? kd : 0;
          const int l = t_budget(h, lo.c2, __popc(pq & ~gm), rem) * sp.tdiv;
          dead = T > l;
          if constexpr (NQ == 3) {
            lim = l;
            tcl = (int)(w >> 24) - 1;
          }
        }
      }
      w2m |= gballot<GS>(c2) << b0;
      w3m |= gballot<GS>(c3) << b0;
      dm |= gballot<GS>(dead) << b0;
    }
    // (a split whose share of the candidates is empty has gbeg >= gend, and gbeg may lie beyond bit 63)
    const uint64_t range = gbeg >= gend ? 0ull : (gend - gbeg < 64 ? (1ull << (gend - gbeg)) - 1 : ~0ull) << gbeg;
    w2m &= range;
    w3m &= range & ~w2m;
    const uint64_t evalm = range & ~w2m & ~w3m;
    dm &= evalm;
    uint64_t todo = evalm & ~dm, alivem = 0, rarem = 0;      // children alive; found or overflowed (their status is written)
    uint32_t settled = (uint32_t)__popcll(dm);
    // n = 3: the status of candidate `lane` as far as the windows decide it
    int wst = ST_DEAD;
    const uint32_t nw2 = (uint32_t)__popcll(w2m), nw3 = (uint32_t)__popcll(w3m), nev = (uint32_t)__popcll(evalm);
    if constexpr (NQ == 3) wst = (w2m >> lane) & 1 ? ST_W2 : (w3m >> lane) & 1 ? ST_W3 : ST_DEAD;
    while (todo) {
      const int g = wuni<NQ>(__ffsll((long long)todo) - 1);
      todo &= todo - 1;
      uint8_t stt;
      uint64_t key = 0;
      uint32_t bw = BW_TUNK;
      {
        // child residual entry (r, c) = sum_m P[r][x_m] ginv[m][lc] (src/cheese.cu:146-174)
        const uint4 hv = tb.head[g];
        const uint32_t hx = (uint32_t)wuni<NQ>((int)hv.x), hw = (uint32_t)wuni<NQ>((int)hv.w);
        int4 s;
        bool of = false;
        int k = pk + wuni<NQ>((int)hv.z);
        const bool fast = STD || ((hw & 1u) && small);
        if (fast) {
          const uint32_t d = tb.term[g * 64 + le];
          const int4 u = P.turned(d & 63u);
          const int m0 = -(int)((d >> 6) & 1u);
          if (hw & 2u) s = make_int4((u.x ^ m0) - m0, (u.y ^ m0) - m0, (u.z ^ m0) - m0, (u.w ^ m0) - m0);
          else {
            int4 v = P.turned((d >> 7) & 63u);
            const int m1 = -(int)((d >> 13) & 1u), on = -(int)((d >> 14) & 1u), o = -m0 - m1;
            v = make_int4(v.x & on, v.y & on, v.z & on, v.w & on);
            s = make_int4((u.x ^ m0) + ((v.x ^ m1) + o), (u.y ^ m0) + ((v.y ^ m1) + o), (u.z ^ m0) + ((v.z ^ m1) + o),
                          (u.w ^ m0) + ((v.w ^ m1) + o));
          }
        } else {
          const DevGate &dg = sp.gates[g];
          int lc = (c >> dg.q[0]) & 1;
          if (dg.nq > 1) lc |= ((c >> dg.q[1]) & 1) << 1;
          if (dg.nq > 2) lc |= ((c >> dg.q[2]) & 1) << 2;
          const int cb = c & ~dg.mask;
          auto source = [&](int m) {
            int x = cb | ((m & 1) << dg.q[0]);
            if (dg.nq > 1) x |= ((m >> 1) & 1) << dg.q[1];
            if (dg.nq > 2) x |= ((m >> 2) & 1) << dg.q[2];
            return P.entry(r * N + x);
          };
          if (dg.unit && small) {
            int4 acc = make_int4(0, 0, 0, 0);
            for (int m = 0; m < dg.L; m++) {
              const int p = dg.ph[m * dg.L + lc];
              if (p < 0) continue;
              const int4 t = zrot(source(m), p);
              acc.x += t.x; acc.y += t.y; acc.z += t.z; acc.w += t.w;
            }
            s = acc;
          } else {
            long long va = 0, vb = 0, vc = 0, vd = 0;
            for (int m = 0; m < dg.L; m++) {
              const int4 gm = dg.inv[m * dg.L + lc];
              if (zzero(gm)) continue;
              const int4 v = source(m);
              va += (long long)v.x * gm.x - (long long)v.y * gm.w - (long long)v.z * gm.z - (long long)v.w * gm.y;
              vb += (long long)v.x * gm.y + (long long)v.y * gm.x - (long long)v.z * gm.w - (long long)v.w * gm.z;
              vc += (long long)v.x * gm.z + (long long)v.y * gm.y + (long long)v.z * gm.x - (long long)v.w * gm.w;
              vd += (long long)v.x * gm.w + (long long)v.y * gm.z + (long long)v.z * gm.y + (long long)v.w * gm.x;
            }
            of = va != (int)va || vb != (int)vb || vc != (int)vc || vd != (int)vd;
            s = make_int4((int)va, (int)vb, (int)vc, (int)vd);
          }
        }
        if (!fast && gany<GS>(of)) stt = ST_OVF;
        else {
          // parents that are children themselves are normalised, which a permutation of unit entries leaves them
          if (!(g1 != 255 && fast && (hw & 2u) && k == pk))
            while (k > 0 && gall<GS>(zhalf(s))) { s = zdown(s); k--; }
          const uint64_t nzb = gballot<GS>(!zzero(s));
          // the goal's entries are read only for a child with the goal's exponent and nonzero pattern
          if (STD ? k == 0 && nzb == ident_mask<NQ>() && gall<GS>(s.x == (r == c) && !(s.y | s.z | s.w))
                  : k == sp.gk && nzb == sp.goalnz && gall<GS>(zeq(s, sp.goal[le])))
            stt = ST_FOUND;
          else {
            bool alive = true;
            if (bounds) {
              int hh, supp = 0, c2 = 0;
              if (lite) hh = k;
              else {
                const int hs = h_struct<NQ>(nzb), gm = (int)((hx >> 8) & 7u);
                hh = k > hs ? k : hs;
                supp = __popc((pq & ~gm) | support_mask<NQ>(s, le, nzb, gm));
              }
              // Bracket the child's bounds from its parent's: the T bound moves by at most the gate's transfer-
              // matrix exponent tdel (Clifford gates keep it), each cut need drops by at most its cdel.  The
              // bound combination is monotone in T and in the cut bound, so the brackets settle most children
              // before the cut ranks and the T transform are computed.
              const int tdel = (int)(hx & 255u);
              const bool tpar = tparent && tdel != 255;
              const int Tp = (int)(pbw & BW_TUNK);
              // a sibling of the same T-bound class already has its exact bound (it is this child's too) or a
              // lower bound
              const int tc = (int)(hx >> 24) - 1;
              const bool tcached = tc >= 0 && ((tc_ok >> tc) & 1);
              const int tcv = tcached ? (int)((tc_val >> (8 * tc)) & 0xff) : 0;
              const bool tcex = tcached && ((tc_ex >> tc) & 1);
              const bool tknown = (tpar && tdel == 0) || tcex;
              const int Tbr = STD && NQ == 3 && cutlow ? (int)gget<GS>((uint32_t)tlo, g) : tpar ? (Tp > tdel ? Tp - tdel : 0) : 0;
              int T = tcex ? tcv : (Tbr > tcv ? Tbr : tcv);    // exact if tknown, else a lower bound
              bool texact = tknown;
              CutLow lo{0, 0, 0};
              if (cutlow) {
                if constexpr (NQ == 3) lo = CutLow{gget<GS>(cl.low, g), (int)gget<GS>((uint32_t)cl.idx, g), (int)gget<GS>((uint32_t)cl.c2, g)};
                else lo = cut_low<NQ, STD>(sp, scx, pneeds, hv.y);
              }
              // alive exactly when T / tdiv, rounded up, is at most t_budget: T <= t_budget * tdiv
              if (T > t_budget(hh, lo.c2, supp, rem) * sp.tdiv) alive = false;
              else {
                if (!lite) {
                  uint32_t needs = pneeds;
                  const uint32_t keepc = (pbw & BW_CUTS) ? hw >> 8 : 0u;
                  const CutStop cst{cutlow && (STD || sp.have_table), lo.low, lo.idx, T, hh, supp, rem};
                  c2 = cx_bound<NQ, STD>(s, le, sp, scx, scsrc, keepc, small, cst, needs, n_cuts);
                  bw = (needs << 8 & ~BW_CUTS) | (STD || sp.ncuts <= BW_MAXCUTS ? BW_CUTS : 0u) | BW_TUNK;
                }
                const int tmax = t_budget(hh, c2, supp, rem) * sp.tdiv;
                if (T > tmax) alive = false;
                else if (!texact && tpar && rem <= 1 && Tp + tdel <= tmax) {
                  // alive whatever the exact T; its children (budget 0) need no inherited T bound
                  alive = true;
                } else if (!texact) {
                  n_t++;
                  if (STD || NQ + k <= 16) {
                    // the f = 0 part, then the flip-pair passes (odd first) while the lower bound leaves the child
                    // alive: at T bound T it is alive exactly when T <= tmax
                    uint32_t np = 0;
                    T = t_bound16s<NQ>(st, s, k, le, T, tmax, np, texact);
                    n_tp += np;
                  } else {
                    T = wuni<NQ>(t_bound_any<NQ>(s, k, le));
                    texact = true;
                  }
                  if (tc >= 0 && T < 255 && (texact || !tcached || T > tcv)) {
                    tc_val = (tc_val & ~(0xffull << (8 * tc))) | (uint64_t)T << (8 * tc);
                    tc_ok |= 1u << tc;
                    if (texact) tc_ex |= 1u << tc;
                    // siblings of the class that this bound puts over their budget (by the parent's bounds) are dead
                    if constexpr (NQ == 3) {
                      const uint64_t sib = gballot<GS>(tcl == tc && T > lim) & todo;
                      if (sib) {
                        todo &= ~sib;
                        settled += (uint32_t)__popcll(sib);
                      }
                    }
                  }
                  alive = T <= tmax;
                }
              }
              if (alive && texact && T < (int)BW_TUNK) bw = (bw & ~BW_TUNK) | (uint32_t)T;
            }
            if (alive && keep) {
              if constexpr (NQ == 3) {
                int image = 0;
                key = class_key3(s, k, lane, spos, tb.kt.adm, cjm, image);
                if (STD || sp.ncuts <= BW_IMAGE_CUTS) bw |= (uint32_t)image << BW_IMAGE;
              } else {
                key = class_key<NQ>(s, k, le, sp);
              }
              key ^= (uint64_t)inst * 0x9e3779b97f4a7c15ull;
            }
            stt = alive ? ST_ALIVE : ST_DEAD;
          }
        }
      }
      if (stt == ST_ALIVE) {
        alivem |= 1ull << g;
        if (keep && le == 0) { a.keys[pl * G + g] = key; a.info[pl * G + g] = bw; }
      } else if (stt != ST_DEAD) {
        rarem |= 1ull << g;
        if (le == 0) {
          a.status[pl * G + g] = stt;
          atomicAdd(&tl[stt], 1u);
          if (stt == ST_FOUND) atomicMin(&icnt[(size_t)inst * IC_N + IC_FIRST], (unsigned long long)((a.off + pl) * G + g));
        }
      }
    }
    // the children's status, one candidate per lane, and their tallies
    for (int b0 = 0; b0 < G; b0 += GS) {
      const int g = b0 + le;
      const bool mine = g >= gbeg && g < gend && !((rarem >> g) & 1);
      const int st_w = NQ == 3 ? wst : (w2m >> g) & 1 ? ST_W2 : (w3m >> g) & 1 ? ST_W3 : ST_DEAD;
      if (mine) a.status[pl * G + g] = (uint8_t)((alivem >> g) & 1 ? (keep ? ST_ALIVE : ST_LAST) : st_w);
    }
    const uint32_t nal = (uint32_t)__popcll(alivem), nrare = (uint32_t)__popcll(rarem);
    n_eval += nev;
    n_pre += settled;
    if (!lite && bounds) n_cheap += nev - settled - nrare;
    if (keep) n_keys += nal;
    if (le == 0) {
      if (nw2) atomicAdd(&tl[ST_W2], nw2);
      if (nw3) atomicAdd(&tl[ST_W3], nw3);
      if (nal) atomicAdd(&tl[ST_ALIVE], nal);
      if (const uint32_t dead = nev - nal - nrare) atomicAdd(&tl[ST_DEAD], dead);
    }
    __builtin_amdgcn_wave_barrier();
  }
  // the block's counts: groups that ended in the first group's instance add up in LDS (a block's groups work on
  // neighbouring parents, so nearly always all of them), the others add to the counters themselves
  __shared__ uint32_t btally[8], bstage[SG_N];
  __shared__ int binst;
  if (threadIdx.x < 8) btally[threadIdx.x] = bstage[threadIdx.x] = 0;
  if (threadIdx.x == 0) binst = cur;
  __syncthreads();
  if (le == 0 && cur >= 0 && cur == binst)
    for (int i = 0; i <= ST_OVF; i++)
      if (const uint32_t v = tl[i]) { atomicAdd(&btally[i], v); tl[i] = 0; }
  flush();
  if (le == 0) {
    const uint32_t n[SG_N - 1] = {n_eval, n_pre, n_t, n_cheap, n_cuts, n_keys, n_tp};     // one copy per group
#pragma unroll
    for (int i = 0; i < SG_N - 1; i++) if (n[i]) atomicAdd(&bstage[i], n[i]);
  }
  __syncthreads();
  if (threadIdx.x < 8) {
    const int i = threadIdx.x;
    if (i <= ST_OVF && btally[i]) atomicAdd(&icnt[(size_t)binst * IC_N + slot_of(i)], (unsigned long long)btally[i]);
    if (bstage[i]) atomicAdd(&a.stage[(blockIdx.x & (NSTRIPE - 1)) * SG_N + i], (unsigned long long)bstage[i]);
  }
}

struct FlagAlive {      // survivors of a chunk that become parents, in child order
  const uint8_t *status;
  __device__ bool operator()(long long i) const { return status[i] == ST_ALIVE; }
};
struct FlagKept {       // kept survivors (k_fill_kept leaves out those of searches that ended)
  const uint8_t *kept;
  __device__ bool operator()(long long i) const { return kept[i] != 0; }
};

// Survivors of a chunk -> level survivor list (child index in the level, class key, bound word).  boff: the tiles' offsets
// from the survivors *out0 of the chunks before; with tot the tiles' counts, the chunk being the level's only one, and
// the total goes to *tot.  boff null: one tile.
struct AliveOut {
  const uint64_t *keys;
  const uint32_t *info;
  long long child0;
  uint64_t *surv_o, *surv_key;
  uint32_t *surv_bw;
};
__global__ __launch_bounds__(CT_THREADS) void k_scatter_alive(FlagAlive f, long long n, const unsigned long long *boff, AliveOut o,
                                                              const unsigned long long *out0, unsigned long long *tot,
                                                              const unsigned long long *nd) {
  n = dev_n(n, nd);
  const unsigned long long pos = !boff ? 0 : tot ? tile_offset(boff, blockIdx.x) : *out0 + boff[blockIdx.x];
  const uint32_t c = tile_compact(f, (long long)blockIdx.x * CT_TILE, n, pos, [&](long long x, unsigned long long p) {
    o.surv_o[p] = (uint64_t)(o.child0 + x);
    o.surv_key[p] = o.keys[x];
    o.surv_bw[p] = o.info[x];
  });
  if (tot && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1) *tot = pos + c;
}

// the level's survivor count grows by a chunk's total (the scan's last entry)
__global__ void k_add_total(unsigned long long *acc, const unsigned long long *tot) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *acc += *tot;
}

// ------------------------------------------------------------------------------------------------------
// segmented dedupe over the sorted survivors: runs of equal 32-bit key prefix are partitioned into exact
// classes, keeping the smallest survivor rank (= lexicographically first prefix) of each class
// (src/cheese.cu:1334-1343, :1046-1065)
// Every survivor of a search that continues after this level (no circuit, no overflow) starts kept: a sequential fill;
// setting kept[v[i]] in the dedupe would scatter byte writes over the array.  (It runs after the level's expansion has read
// the goal flags, before the gather sets them for the next level: gflag, when given, is cleared here.)
struct ActiveArgs {
  const unsigned long long *icnt;   // the expansion's per-slot counters, in nstr stripes
  int nstr, ns, G;
  const uint64_t *surv_o;
  const uint32_t *pinst;
};
constexpr int ACT_LDS = 1024;       // slots whose state a block keeps in LDS; beyond it is read per survivor
__device__ __forceinline__ bool slot_ended(const ActiveArgs &a, int s) {
  unsigned long long x = 0;
  for (int j = 0; j < a.nstr; j++) {
    const unsigned long long *c = a.icnt + ((size_t)j * a.ns + s) * IC_N;
    x |= c[IC_FOUND] | c[IC_OVF];
  }
  return x != 0;
}
__global__ __launch_bounds__(256) void k_fill_kept(uint8_t *kept, long long n, const unsigned long long *nd, ActiveArgs a,
                                                   uint32_t *gflag) {
  __shared__ uint32_t ended[ACT_LDS];
  n = dev_n(n, nd);
  const bool lds = a.ns <= ACT_LDS;
  if (lds) {
    for (int s = threadIdx.x; s < a.ns; s += blockDim.x) ended[s] = 0;
    __syncthreads();
    for (int i = threadIdx.x; i < a.ns * a.nstr; i += blockDim.x) {
      const unsigned long long *c = a.icnt + (size_t)i * IC_N;
      if (c[IC_FOUND] | c[IC_OVF]) atomicOr(&ended[i % a.ns], 1u);
    }
    __syncthreads();
  }
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, stride = (long long)gridDim.x * blockDim.x;
  for (long long i = i0; i < n; i += stride) {
    const int s = (int)a.pinst[a.surv_o[i] / (uint64_t)a.G];
    kept[i] = !(lds ? ended[s] != 0 : slot_ended(a, s));
  }
  if (gflag)
    for (long long i = i0; i < a.ns; i += stride) gflag[i] = 0u;
}

struct DedupeArgs {
  const uint32_t *k, *v;          // sorted key prefixes and survivor ranks
  long long n;
  const uint64_t *surv_o, *surv_key;
  const uint32_t *surv_bw;
  const int4 *res;                // parents' residuals
  const int *pk;
  uint8_t *kept;
  unsigned long long *cnt;
  const uint32_t *pinst;          // parents' instance slots (null: one instance)
  const unsigned long long *nd;   // survivors read on the device (captured step), or null
};
constexpr int MAXREP = 32, MAXSYM = 32;

// the candidates' entry descriptors and exponents, copied into LDS by a block that forms children with child_terms
struct ChildTab {
  uint16_t desc[MAXG * 64];
  uint8_t ik[MAXG];
};
__device__ __forceinline__ void load_child_tab(ChildTab &t, const KSpec &sp) {
  const SpecTabs *g = (const SpecTabs *)sp.ktab;
  for (int i = threadIdx.x; i < sp.G * 8; i += blockDim.x) ((uint4 *)t.desc)[i] = ((const uint4 *)g->sdesc)[i];
  for (int i = threadIdx.x; i < sp.G; i += blockDim.x) t.ik[i] = (uint8_t)g->level.head[i].z;
}

template <int NQ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(NQ > 1 ? 5 : 1)))
void k_dedupe_runs(KSpec sp, DedupeArgs a) {
  constexpr int N = 1 << NQ, E = N * N, GS = E, CPW = 64 / GS;
  constexpr int GPB = 256 / GS;     // groups per block
  __shared__ uint64_t rep_key[GPB][MAXREP], rep_o[GPB][MAXREP];
  __shared__ uint32_t rep_inst[GPB][MAXREP];
  __shared__ uint8_t spos[MAXSYM * E];
  __shared__ int4 rep_img[GPB][2][E];     // images of the first two representatives' residuals (same_class_image)
  __shared__ __align__(16) ChildTab ct;
  load_child_tab(ct, sp);
  // the symmetry group's entry maps, staged once per block (the class test tries the elements in order)
  const int nsym = sp.nsym < MAXSYM ? sp.nsym : MAXSYM;
  const bool lds_sym = nsym == sp.nsym;
  uint32_t cjm = 0;
  for (int i = threadIdx.x; i < nsym * E; i += blockDim.x) {
    const int y = i / E, e = i % E;
    spos[i] = (uint8_t)(sp.symperm[y * N + (e >> NQ)] * N + sp.symperm[y * N + (e & (N - 1))]);
  }
  for (int y = 0; y < nsym; y++) cjm |= (uint32_t)(sp.symconj[y] != 0) << y;
  __syncthreads();
  const int lane = threadIdx.x & 63, le = lane & (GS - 1), slot = lane / GS;
  const int grp = (threadIdx.x >> 6) * CPW + slot;
  const long long wave = wave_index();
  const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
  const long long n = dev_n(a.n, a.nd);
  const uint64_t G = (uint64_t)sp.G;
  constexpr uint64_t ALL = GS == 64 ? ~0ull : (1ull << GS) - 1;
  // A lane group takes up to GS sorted positions at a time and deduplicates the runs of equal prefixes that start there, lane
  // le holding position le's rank, child, key, parent exponent and slot: the chain of five dependent loads from a run to
  // its members' parents is waited for once a tile, and each member then waits on one load (its parent's residual), issued
  // while the member before it is compared, be it of another run.  (One run at a time, from a list of the runs: the
  // budget-14 proof's dedupe 20.4 ms under the tracer, here 15.0.)
  // A run is almost always one class: its members are each rebuilt once and compared with the first representative, of which
  // (and of the second) an image stays in LDS.  A member's smallest image is known from its class key, so one comparison
  // settles it where trying the group's elements in turn took six or seven; its entries come straight from its parent in
  // global memory.  (With the members' parents staged in LDS, gate tables in global memory and the elements tried in
  // turn it took another 8 ms.)
  // Smaller tiles where there are not enough positions for all groups: a small level's dedupe is as long as its longest chain.
  int tn = 4;
  while (tn < GS && tn * nwaves * CPW < n) tn <<= 1;
  for (long long t0 = (wave * CPW + slot) * tn; t0 < n; t0 += nwaves * CPW * tn) {
    long long j0 = t0;
    uint32_t key = 0;             // of the run that crosses the tile's end, once it is walked
    bool crossing = false;
    int nrep = 0, head = -1;
    int ck0 = 0, ck1 = 0;
    for (;;) {
      const long long jj = j0 + le;
      const bool valid = jj < n && (crossing || le < tn);
      const uint32_t kj = valid ? a.k[jj] : 0u;
      uint64_t heads = 0, left, over = 0;       // over: the run that the tile's last position shares with the next tile
      bool in;
      if (!crossing) {
        const bool first = valid && (jj == 0 || a.k[jj - 1] != kj), more = valid && jj + 1 < n && a.k[jj + 1] == kj;
        heads = gballot<GS>(first);
        const uint64_t cont = gballot<GS>(more);
        if (!heads) break;                      // the tile lies within a run of an earlier one
        const int h0 = __ffsll((long long)heads) - 1;
        if ((cont >> (tn - 1)) & 1) over = ALL & ~((1ull << (63 - __clzll((long long)heads))) - 1);
        in = le >= h0 && !((over >> le) & 1) && (more || !first) && valid;
      } else in = valid && kj == key;
      uint32_t m_rank = 0, m_inst = 0, m_img = 0;
      uint64_t m_o = 0, m_key = 0;
      int m_pk = 0;
      if (in) {
        m_rank = a.v[jj];
        m_o = a.surv_o[m_rank];
        m_key = a.surv_key[m_rank];
        m_img = NQ == 3 && sp.ncuts <= BW_IMAGE_CUTS ? (a.surv_bw[m_rank] >> BW_IMAGE) & 15u : 0u;
        const long long pi = (long long)(m_o / G);
        m_pk = a.pk[pi];
        m_inst = a.pinst ? a.pinst[pi] : 0u;
      }
      const uint64_t inb = gballot<GS>(in);
      left = inb;
      if (!crossing) {
        // runs of two: only members that share their whole key are looked at (the sort brings together what agrees in
        // part of it)
        const uint64_t up = (uint64_t)(uint32_t)__shfl_down((int)(m_key >> 32), 1, GS) << 32 | (uint32_t)__shfl_down((int)m_key, 1, GS);
        const uint64_t eq = gballot<GS>(in && m_key == up);
        const uint64_t two = heads & inb & ~(heads >> 1) & (heads >> 2 | ~(inb >> 2));
        const uint64_t apart = two & ~eq;
        left &= ~(apart | apart << 1);
      }
      auto terms = [&](int q) {
        const uint64_t o = gget64<GS>(m_o, q);
        return child_terms<NQ>(a.res + (long long)(o / G) * E, ct.desc[(int)(o % G) * 64 + le], le);
      };
      ChildTerms next{};
      if (left) next = terms(__ffsll((long long)left) - 1);
      while (left) {
        const int q = __ffsll((long long)left) - 1;
        left &= left - 1;
        if (!crossing) {
          const int h = 63 - __clzll((long long)(heads & ((2ull << q) - 1)));
          if (h != head) { head = h; nrep = 0; }
        }
        const uint32_t rank = gget<GS>(m_rank, q), inst = gget<GS>(m_inst, q);
        const uint64_t o = gget64<GS>(m_o, q), key64 = gget64<GS>(m_key, q);
        const int pk = (int)gget<GS>((uint32_t)m_pk, q), img = (int)gget<GS>(m_img, q);
        const int g = (int)(o % G);
        const ChildTerms cur = next;
        if (left) next = terms(__ffsll((long long)left) - 1);
        int4 s;
        int ks;
        if (!child_of<NQ>(cur, ct.desc[g * 64 + le], ct.ik[g], pk, s, ks))
          make_child<NQ>(a.res + (long long)(o / G) * E, pk, sp.gates[g], le, s, ks);
        bool dup = false;
        for (int r = 0; r < nrep && !dup; r++) {
          if (rep_key[grp][r] != key64 || rep_inst[grp][r] != inst) continue;
          if (r < 2 && lds_sym) {
            dup = same_class_image<NQ>(s, ks, rep_img[grp][r], r ? ck1 : ck0, img, le, spos, cjm, nsym);
          } else {
            int4 b;
            int kb;
            const uint64_t ro = rep_o[grp][r];
            const long long rpi = (long long)(ro / G);
            make_child<NQ>(a.res + rpi * E, a.pk[rpi], sp.gates[(int)(ro % G)], le, b, kb);
            dup = lds_sym ? same_class_lds<NQ>(s, ks, b, kb, le, spos, cjm, nsym) : same_class<NQ>(s, ks, b, kb, le, sp);
          }
        }
        if (dup) { if (le == 0) a.kept[rank] = 0; }
        else if (nrep < MAXREP) {
          if (le == 0) {
            rep_key[grp][nrep] = key64;
            rep_o[grp][nrep] = o;
            rep_inst[grp][nrep] = inst;
          }
          if (nrep < 2) {
            rep_img[grp][nrep][spos[img * GS + le]] = (cjm >> img) & 1 ? zconj(s) : s;
            if (nrep == 0) ck0 = ks;
            else ck1 = ks;
          }
          nrep++;
        } else if (le == 0) atomicAdd(&a.cnt[C_REPOVF], 1ull);
        __builtin_amdgcn_wave_barrier();
      }
      if (!crossing) {
        if (!over) break;
        crossing = true;                        // from its head, GS members at a time
        nrep = 0;
        const int h = __ffsll((long long)over) - 1;
        j0 = t0 + h;
        key = a.k[j0];
      } else if (inb == ALL) j0 += GS;
      else break;
    }
  }
}

// T columns of a frontier node: the columns of its residual's Pauli transfer matrix (Paulis, X bits then Z bits) known to
// attain its T bound, 0 when none is known.  The gather takes them from the parent where the gate only permutes columns, or
// where the bound is the parent's; k_tcols forms those of the others.
struct GatherArgs {
  const uint32_t *kidx;           // kept survivor ranks, in order
  long long nk;
  const uint64_t *surv_o;
  const int4 *res;
  const int *pk;
  const uint8_t *g1;
  int4 *res_next;
  int *pk_next;
  uint8_t *g1_next, *g2_next;
  uint32_t *tree_par;
  uint8_t *tree_gate;
  const uint32_t *pinst;          // parents' instance slots (null: one instance)
  uint32_t *inst_next;
  const uint32_t *surv_bw;        // bound words of the survivors
  uint32_t *pb_next;
  const unsigned long long *nkd;  // kept count read on the device (captured step), or null
  uint32_t *gflag;                // per slot: set when a kept child has a goal child (null: not tracked)
  int tn;                         // kept nodes per wave tile (a multiple of the nodes per wave, at most 64)
};

// next frontier: tree node, window state and materialised residual of every kept child.  A wave takes tiles
// of a.tn consecutive kept nodes: one lane per node resolves the node's index chain (kept rank -> survivor ->
// parent and gate) and writes its small fields, then the lane groups build the tile's residuals from the
// parents, with the chain already in registers.
// It is bound by memory (1 KB read and written per node at n = 3): 11.2 million nodes of the Toffoli budget-14 proof take
// 5.9 ms, 4.9 at the rate of a large copy; 11.3 with gate tables and goal pre-images read from global memory per node.
template <int NQ>
__global__ __launch_bounds__(256) void k_gather(KSpec sp, GatherArgs a, const uint32_t *pb, const uint64_t *tm, uint64_t *tm_next) {
  constexpr int N = 1 << NQ, E = N * N, GS = E, CPW = 64 / GS;
  const int lane = threadIdx.x & 63, le = lane & (GS - 1), slot = lane / GS;
  const long long wave = wave_index();
  const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
  const long long nk = dev_n(a.nk, a.nkd);
  const int tn = a.tn;
  __shared__ __align__(16) ChildTab ct;
  load_child_tab(ct, sp);
  __shared__ __align__(16) uint8_t col_src[NQ == 3 ? MAXG * 64 : 16];
  if (NQ == 3 && tm)
    for (int i = threadIdx.x; i < sp.G * 4; i += blockDim.x) ((uint4 *)col_src)[i] = ((const uint4 *)((const SpecTabs *)sp.ktab)->col_src)[i];
  __syncthreads();
  // goal pre-images, one candidate per lane (n = 3: every candidate)
  const int xgk = NQ == 3 && a.gflag && lane < sp.G ? sp.xgk[lane] : -1;
  const uint64_t xgm = NQ == 3 && a.gflag && lane < sp.G ? sp.xgm[lane] : 0ull;
  const uint32_t bwkeep = NQ == 3 && sp.ncuts <= BW_IMAGE_CUTS ? ~(15u << BW_IMAGE) : ~0u;
  for (long long tb = wave * tn; tb < nk; tb += nwaves * tn) {
    const long long pl = tb + lane;
    uint32_t pi_l = 0, bw_l = 0;
    uint64_t tm_l = 0;             // the parent's T columns, where they say something of the node's
    int g_l = 0, gp_l = 255, pk_l = 0;
    if (lane < tn && pl < nk) {
      const uint32_t kid = a.kidx[pl];
      const uint64_t o = a.surv_o[kid];
      pi_l = (uint32_t)(o / (uint64_t)sp.G);
      g_l = (int)(o % (uint64_t)sp.G);
      bw_l = a.surv_bw[kid] & bwkeep;
      gp_l = a.g1[pi_l];
      pk_l = a.pk[pi_l];
      if (NQ == 3 && tm && !((pb[pi_l] ^ bw_l) & BW_TUNK) && (bw_l & BW_TUNK) != BW_TUNK) tm_l = tm[pi_l];
      if (NQ == 3 && !tm && tm_next) tm_next[pl] = 0;     // no node has any yet
      a.g1_next[pl] = (uint8_t)g_l;
      a.g2_next[pl] = (uint8_t)gp_l;
      a.tree_par[pl] = pi_l;
      a.tree_gate[pl] = (uint8_t)g_l;
      a.inst_next[pl] = a.pinst ? a.pinst[pi_l] : 0u;
    }
    // a node's parent entries are on the way while the node before it is finished
    auto terms = [&](int src) {
      const uint32_t pi = (uint32_t)__shfl((int)pi_l, src);
      const int g = __shfl(g_l, src);
      ChildTerms t{};
      if (src < tn && tb + src < nk) t = child_terms<NQ>(a.res + (long long)pi * E, ct.desc[g * 64 + le], le);
      return t;
    };
    ChildTerms next = terms(slot);
    for (int j = 0; j < tn; j += CPW) {
      const int src = j + slot;
      const long long pi = (long long)(uint32_t)__shfl((int)pi_l, src);
      const int g = __shfl(g_l, src), gp = __shfl(gp_l, src), pk = __shfl(pk_l, src);
      const uint32_t bwp = (uint32_t)__shfl((int)bw_l, src);
      const long long p = tb + src;
      const ChildTerms cur = next;
      if (j + CPW < tn) next = terms(j + CPW + slot);
      if (src >= tn || p >= nk) continue;
      int4 s;
      int k;
      if (!child_of<NQ>(cur, ct.desc[g * 64 + le], ct.ik[g], pk, s, k))
        make_child<NQ>(a.res + pi * E, pk, sp.gates[g], le, s, k);
      a.res_next[p * E + le] = s;
      // goal child: the node equals the pre-image of a candidate its windows allow.  One lane per candidate
      // filters by exponent and nonzero pattern; the few that pass are compared exactly.
      bool adj = false;
      if (a.gflag) {
        const uint64_t nzb = gballot<GS>(!zzero(s));
        for (int b0 = 0; b0 < sp.G && !adj; b0 += GS) {
          const int x = b0 + le;
          uint64_t cm = NQ == 3 ? gballot<GS>(xgk == k && xgm == nzb)
                                : gballot<GS>(x < sp.G && sp.xgk[x] == k && sp.xgm[x] == nzb);
          while (cm && !adj) {
            const int xx = b0 + __builtin_ctzll(cm);
            cm &= cm - 1;
            bool ok = sp.bad2[g * sp.G + xx] == 0;
            if (ok && gp != 255) {
              const uint32_t tri = ((uint32_t)gp * sp.G + g) * sp.G + xx;
              ok = ((sp.bad3[tri >> 5] >> (tri & 31)) & 1) == 0;
            }
            if (ok) adj = gall<GS>(zeq(s, sp.xg[xx * E + le]));
          }
        }
      }
      if (NQ == 3 && tm) {
        const uint64_t pt = gget64<64>(tm_l, src);
        const uint8_t from = pt ? col_src[g * 64 + lane] : (uint8_t)255;
        const uint64_t t = gballot<64>(from < 64 && ((pt >> (from & 63)) & 1));
        if (le == 0) tm_next[p] = t;
      }
      if (le == 0) {
        a.pk_next[p] = k;
        a.pb_next[p] = bwp | (adj ? BW_GOAL : 0u);
        if (adj) a.gflag[a.pinst ? a.pinst[pi] : 0u] = 1u;
      }
    }
  }
}

// T columns of the nodes of a frontier that have none and whose T bound is known (n = 3; n + k <= 16), unless no T gate can
// follow in the budget or the search ends at the next level: one pass of the
// bound's transform, the one whose parity its valuation v has, and per column the bit that makes it v.  Only Paulis with
// an X part on the residual's left count (flip pairs f >= 8): there the bit that the pairs leave out is one of the rows, and
// the columns' bits are the low three of the transform's index.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void k_tcols(KSpec sp, const int4 *res, const int *pk, const uint32_t *pb,
                                                                                    const uint32_t *inst, const int *rem, const uint32_t *gflag,
                                                                                    uint64_t *tm, long long n) {
  constexpr int NQ = 3, H = 32;
  __shared__ __align__(1024) uint4 stage[2 * TS_STRIDE];
  const int lane = threadIdx.x & 63;
  const TStage st{(char *)stage, (threadIdx.x & ~63u) << 4};
  const int f = lane == 0 ? 1 : lane, j = 31 - __clz(f);
  uint32_t vb[2 * NQ - 1];
#pragma unroll
  for (int b = 0; b < 2 * NQ - 1; b++) vb[b] = (b >= j ? 32u : 16u) << b;
  const uint32_t fo = (uint32_t)f << 4;
  const long long nwaves = ((long long)gridDim.x * blockDim.x) >> 6;
  // 16 nodes a wave and turn: with 64, a frontier of some ten thousand nodes left most of the chip idle
  for (long long t0 = wave_index() * 16; t0 < n; t0 += nwaves * 16) {
    int v_l = 0;
    if (lane < 16 && t0 + lane < n && tm[t0 + lane] == 0) {
      const uint32_t bw = pb[t0 + lane], nd = (bw & BW_NEEDS) >> 8;
      const int T = (int)(bw & BW_TUNK), k = pk[t0 + lane];
      if (T != (int)BW_TUNK && T > 0 && (bw & BW_CUTS) && NQ + k <= 16) {
        const int c2 = sp.cxtable[(nd & 7u) + 3 * ((nd >> 3) & 7u) + 9 * ((nd >> 6) & 7u)];
        const uint32_t i = inst[t0 + lane];
        if (!(gflag && gflag[i]) && t_budget(k, c2, 0, rem[i] - 1) * sp.tdiv >= T - 1) v_l = 2 * (NQ + k) - T;
      }
    }
    uint64_t todo = gballot<64>(v_l > 0);
    while (todo) {
      const int x = __ffsll((long long)todo) - 1;
      todo &= todo - 1;
      const int v = (int)gget<64>((uint32_t)v_l, x), pass = v & 1, m = (v - 2 + pass) >> 1;
      const int4 s = res[(t0 + x) * 64 + lane];
      __builtin_amdgcn_wave_barrier();
      t_stage_x<NQ>(st, s, lane);
      t_stage_p<NQ>(st, s, lane, pass);
      __builtin_amdgcn_wave_barrier();
      uint32_t at = st.group;
      asm volatile("" : "+v"(at));
      u16x2 q[H];
#pragma unroll
      for (int t = 0; t < H; t++) {
        if (t) at ^= vb[t & 1 ? 0 : t & 2 ? 1 : t & 4 ? 2 : t & 8 ? 3 : 4];
        const uint2 xv = *(const uint2 *)(st.lds + 16 * TS_STRIDE + (at ^ fo));
        const uint4 mm = *(const uint4 *)(st.lds + at);
        const u16x2 x01 = as16(xv.x), x23 = as16(xv.y);
        q[t ^ (t >> 1)] = x01.xx * as16(mm.x) + x01.yy * as16(mm.y) + x23.xx * as16(mm.z) + x23.yy * as16(mm.w);
      }
#pragma unroll
      for (int h = 1; h < H / 2; h <<= 1)
#pragma unroll
        for (int i = 0; i < H; i++)
          if (!(i & h)) {
            const u16x2 a = q[i], b = q[i | h];
            q[i] = a + b;
            q[i | h] = a - b;
          }
      // (the last step as in t_bound16s: no value has a bit below m, so bit m says that one of the column's attains it)
      uint64_t cols = 0;
#pragma unroll
      for (int z = 0; z < 8; z++) {
        uint32_t o = 0;
#pragma unroll
        for (int i = z; i < H / 2; i += 8) {
          const uint32_t a = bits(q[i]), b = bits(q[i | H / 2]);
          o |= (a ^ b) | ((a & b) << 1 & 0xfffefffeu);
        }
        uint64_t on = gballot<64>(((o | o >> 16) >> m) & 1u) & ~0xffull;
        on |= on >> 32;
        on |= on >> 16;
        on |= on >> 8;
        cols |= (on & 0xffull) << (8 * z);
      }
      if (lane == 0) tm[t0 + x] = cols;
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// nodes per gather tile: one per lane group while the launch has enough waves for all of them, up to 64
template <int NQ> static int gather_tile(long long nk) {
  constexpr int CPW = 64 / (1 << (2 * NQ));
  const long long waves = 8192ll * 4;
  long long tn = (nk + waves - 1) / waves;
  tn = (tn + CPW - 1) / CPW * CPW;
  return (int)std::max<long long>(CPW, std::min<long long>(64, tn));
}


// 64-bit class keys -> sortable prefixes and survivor ranks
__global__ void k_init_sort(const uint64_t *key, long long n, int passes, uint32_t *k32, uint32_t *v32,
                            const unsigned long long *nd) {
  n = dev_n(n, nd);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    k32[i] = sort_prefix(key[i], passes);
    v32[i] = (uint32_t)i;
  }
}

// ------------------------------------------------------------------------------------------------------
// host side

// K_STEP: a captured level step (expansion through kept compaction in one graph launch, small levels)
enum { K_EXPAND = 0, K_COMPACT, K_SORT, K_DEDUPE, K_GATHER, K_STEP, K_NFAM };
static const char *k_names[K_NFAM] = {"expand", "compact", "sort", "dedupe", "gather", "level_graph"};

#include "table_join_kernels.h"

}  // namespace chz

namespace chz {
// one search of a batch (searches that share a spec's gate set advance level by level together)
struct BInst {
  int tag = 0, depth = 0, t = 0, slot = 0, root_step = -1;
  bool live = false;
  long long nodes = 0;
  double growth = 0;           // the last level's distinct / parents (0: not known yet)
  int k = 0;                   // the root's sqrt2 exponent and largest coefficient
  uint32_t coef = 0;
  bool reducible = false;      // sqrt2 divides the root's entries below its exponent
  double t0 = 0;
};
struct Pending {               // a search waiting to join the frontier as a root
  int inst, k;
  std::vector<int4> U;
};
}  // namespace chz

struct chz_ctx {
  chz::HostSpec hs;
  chz::SymGroup grp;
  chz_opts opts{};
  int depth = 0;
  int device = 0;
  hipStream_t stream = nullptr;
  chz::KSpec ks{};
  // spec on the device
  chz::DBuf<uint8_t> spec_blob;     // the device tables below, one block
  chz::DBuf<uint8_t> ktab;          // the expansion kernel's LDS tables (LevelTabs)
  chz::DevGate *d_gates = nullptr;
  uint8_t *d_bad2 = nullptr, *d_symperm = nullptr, *d_symconj = nullptr;
  uint32_t *d_bad3 = nullptr;
  int4 *d_goal = nullptr, *d_xg = nullptr;
  uint64_t *d_xgm = nullptr;
  int *d_cx = nullptr, *d_xgk = nullptr;
  // frontier (current and next generation) and the tree of all levels
  chz::DBuf<int4> res[2];
  chz::DBuf<int> pk[2];
  chz::DBuf<uint8_t> g1[2], g2[2];
  chz::DBuf<uint32_t> pb[2];        // bound words (T bound, cut needs) of the frontier's nodes
  chz::DBuf<uint64_t> tm[2];        // their T columns (3 qubits, specialised expansion)
  std::vector<uint32_t *> tree_par;
  std::vector<uint8_t *> tree_gate;
  // per-level work arrays
  chz::DBuf<uint8_t> status, kept;
  chz::DBuf<uint64_t> keys, surv_o, surv_key;
  chz::DBuf<uint32_t> info, surv_bw;
  chz::DBuf<unsigned long long> bcount, hist;
  chz::DBuf<uint32_t> sk[2], sv[2], kidx;
  // batch state: searches, frontier instance slots, per-slot device arrays, queued events
  std::vector<chz::BInst> binst;
  std::vector<chz::Pending> pending;
  std::deque<chz_event> events;
  chz::DBuf<uint32_t> finst[2];
  long long m = 0;             // nodes in the current frontier (buffer cur)
  int cur = 0, gstep = -1, nslots = 0;
  bool shared_steps = false;      // the batch has held more than one search at once (captured steps are used)
  // level control block, uploaded in one copy at the start of every level and read back in one copy:
  // [cnt: C_N counters | stage stripes | icnt: stripes of per-slot IC_N counters | slo, shi: each slot's nodes in the next
  // frontier | d_rem: per-slot budgets | d_keepi: per-slot keep flags]
  chz::DBuf<unsigned long long> ctl;
  unsigned long long *cnt = nullptr, *stage = nullptr, *icnt = nullptr;
  long long *slo = nullptr, *shi = nullptr;
  int *d_rem = nullptr;
  uint8_t *d_keepi = nullptr;
  chz::DBuf<uint32_t> gflag;        // per slot: a node of the current frontier has a goal child
  chz::DBuf<unsigned long long> scan_tmp;
  chz::Pinned pin;                  // staging of the per-level control transfers
  chz::Pinned pin_io;               // what kernels read and write on the host: admitted roots, walked circuits
  chz::Retired retired;             // outgrown buffers, given back when the stream has synchronised
  // captured level steps (one per frontier parity) and the buffer addresses and schedule they were captured with
  struct StepGraph { hipGraphExec_t exec = nullptr; std::vector<uintptr_t> key; };
  StepGraph sgraph[2];
  // expansion schedule per level-size bucket (log2 of the chunk's parents): occupancy variant, grid cap in
  // blocks, candidate-split threshold in waves; chosen by chz_tune, defaults otherwise
  struct Sched { int var = 1, cap = 8192, tw = 4096; };
  Sched sched[32];
  bool tuning = false;
  Sched force;
  std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> tune_ev;   // (bucket, events) per launch
  std::map<void *, size_t> tree_blocks;   // every tree block allocated, with its size
  std::vector<void *> tree_free;          // blocks no live search reaches, ready for reuse
  // measurement
  chz::EventLog ev;
  long k_launch[chz::K_NFAM] = {};
  double k_ms[chz::K_NFAM] = {}, k_work[chz::K_NFAM] = {};
  double k_stage[6] = {};       // expansion stage counts: children past the windows, structural bounds, cut ranks, T bounds,
                                // keys, T-bound passes
  double avg_terms = 1;         // nonzero terms per inverse column, averaged over the candidates
  double avg_qubits = 1;        // qubits per candidate
  bool tcols = false;           // 3 qubits and std_spec: the frontier carries T columns
  bool cols_on = false;         // some node of it may have any
  bool cols_formed = false;     // the candidates' column maps are on the device
  bool std_spec = false;        // what the specialised expansion asks of a spec
  int max_ik = 0;               // the largest sqrt2 exponent of a gate
  bool goal_skip = false;       // every candidate has a goal pre-image: the found-level skip is exact
  // per-level memory planning (chz_batch_set_budget): searches in frontier order; with a budget, a level expands
  // the longest prefix of them whose planned bytes fit, and the rest wait, carried to the next frontier unexpanded
  std::vector<int> forder;
  double mem_budget = 0;
  long long carried_levels = 0;   // search-levels that waited (measurement)
  // --table K: the distance table (built on first use, kept with the context); a context that builds one has
  // gt_filter set (its levels drop classes the table holds and are appended to it) and no goal test
  chz::GTable *gt = nullptr;
  chz::GTable *gt_filter = nullptr;
  bool nogoal = false;
  chz::DBuf<uint64_t> gt_keys, gt_hit;
  chz::DBuf<uint8_t> gt_cost;
  chz::DBuf<unsigned long long> gt_best;
};

namespace chz {

// (the context's stream has synchronised: the blocks go back to the process-wide cache)
static void free_tree(chz_ctx *c) {
  for (auto &kv : c->tree_blocks) dev_pool().put(kv.first, kv.second);
  c->tree_blocks.clear();
  c->tree_free.clear();
  c->tree_par.clear();
  c->tree_gate.clear();
}

// one tree level of n nodes (parents u32, then gates u8) from the block pool
static void tree_alloc(chz_ctx *c, long long n, uint32_t *&tp, uint8_t *&tg) {
  const size_t need = (size_t)std::max<long long>(n, 1) * 5;
  void *blk = nullptr;
  for (size_t i = 0; i < c->tree_free.size(); i++)
    if (c->tree_blocks[c->tree_free[i]] >= need) {
      blk = c->tree_free[i];
      c->tree_free.erase(c->tree_free.begin() + i);
      break;
    }
  if (!blk) {
    size_t got = 0;
    blk = block_get(need + need / 4 + 256, got);
    c->tree_blocks[blk] = got;
  }
  tp = (uint32_t *)blk;
  tg = (uint8_t *)(tp + std::max<long long>(n, 1));
}

// Lane operations of the T bound as implemented, two 16-bit operations to a packed one.  The f = 0 part: per entry 14 16-bit
// operations for |S|^2 = r + y sqrt2 and 1 for each of r and y per transform stage.  One flip-pair pass: for each of the
// 4^n - 1 flip pairs, half of E/2 Z[w] products (8 multiplies and 6 adds of 16 bits), a (2n - 2)-stage transform of E/2
// two-coefficient entries, and in place of the last stage 3 operations for every two of them.
static double t_f0_ops(int nq) {
  const double E = (double)(1 << (2 * nq));
  return E * 7 + 2 * nq * E;
}
static double t_pass_ops(int nq) {
  const double E = (double)(1 << (2 * nq)), H = E / 2;
  return (E - 1) * H * (7 + (2 * nq - 2) + 1.5);
}

// Algorithmic integer operations of one level's expansion, by stage, in 32-bit lane operations (two 16-bit
// operations of the packed T transform count as one); what is done for a parent as a whole is not counted:
//   residual (of the children that form one): per entry, 8 per nonzero term of the gate's inverse column (4 coefficients
//             turned, 4 adds), plus 6 for the sqrt2-divisibility test and 4 for the goal comparison;
//   structural bounds: per entry 4 for the nonzero test, 5 per qubit of the gate for the support comparison;
//   cut rank: per entry 14 per elimination step (2 products, 1 modular subtraction and reduction), two steps, and a third
//             of the F_p image, which a child's ranks share (4 products and one reduction, 9);
//   T bound: t_f0_ops per evaluation, t_pass_ops per flip-pair pass it ran;
//   class key: per entry 9 for each of the two entry hashes; n = 3: 3 sums that choose the symmetries (7 steps and 2 to
//             form a share each) and one image (6 for the summand, two sums), n < 3: every image.
static double expand_ops(const chz_ctx *c, int nq, const unsigned long long *hc) {
  const double E = (double)(1 << (2 * nq));
  const double child = E * (8.0 * c->avg_terms + 10.0), cheap = E * (4.0 + 5.0 * c->avg_qubits), cut = E * (2 * 14.0 + 3.0);
  const double image = 6.0 + 2.0 * (nq == 3 ? 7 : 2 * nq);
  const double key = E * (2 * 9.0 + (nq == 3 ? 3 * 9.0 + image : image * c->ks.nsym));
  return (double)(hc[C_EVAL] - hc[C_PRE]) * child + (double)hc[C_CHEAP] * cheap + (double)hc[C_CUTS] * cut +
         (double)hc[C_NEEDT] * t_f0_ops(nq) + (double)hc[C_TPASS] * t_pass_ops(nq) + (double)hc[C_KEYS] * key;
}


constexpr uint32_t NO_PARENT = 0xffffffffu;
constexpr uint8_t CARRY_GATE = 0xfe;      // tree entry of a node carried unexpanded to the next level

// tree entries of n carried nodes: parent = their index in the level before (first_old + j)
__global__ void k_carry_tree(uint32_t *tp, uint8_t *tg, long long n, long long first_old) {
  for (long long j = (long long)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (long long)gridDim.x * blockDim.x) {
    tp[j] = (uint32_t)(first_old + j);
    tg[j] = CARRY_GATE;
  }
}

// (key prefix, rank) pairs of the survivors in sk[0]/sv[0], equal prefixes together in order of rank.  nd: their number
// is read on the device, n bounds it.
static void sort_survivors(chz_ctx *c, long long n, const unsigned long long *nd, hipStream_t s) {
  for (int b = 0; b < 2; b++) { c->sk[b].need(n); c->sv[b].need(n); }
  if (n <= SS_MAX) {
    hipLaunchKernelGGL(k_sort_small, dim3(1), dim3(SS_THREADS), 0, s, c->surv_key.p, n, c->sk[0].p, c->sv[0].p, nd);
    return;
  }
  const int passes = sort_passes(n), from = passes & 1;
  const long long nb = (n + RS_TILE - 1) / RS_TILE;
  c->hist.need((size_t)nb * 256 + 1);
  c->scan_tmp.need((size_t)nb * 256 / SC_TILE + 4);
  hipLaunchKernelGGL(k_init_sort, dim3(grid_for(n / 64 + 1)), dim3(256), 0, s, c->surv_key.p, n, passes, c->sk[from].p,
                     c->sv[from].p, nd);
  HIPCHK(radix_sort_pairs(c->sk[0].p, c->sv[0].p, c->sk[1].p, c->sv[1].p, n, c->hist.p, c->scan_tmp.p, s, nd, passes));
}

// the survivors of the level's only chunk, in order, their number in C_SURV.  (A gate set without candidates has no
// children: nothing is launched, since an empty grid is an error that the thread's next hipGetLastError would return.)
static void compact_alive(chz_ctx *c, const FlagAlive &fa, long long ncc, const AliveOut &ao, const unsigned long long *dncc,
                          hipStream_t s) {
  if (ncc == 0) return;
  const long long nb = (ncc + CT_TILE - 1) / CT_TILE;
  if (nb > 1)
    hipLaunchKernelGGL(k_flag_count<FlagAlive>, dim3((unsigned)nb), dim3(CT_THREADS), 0, s, fa, ncc, c->bcount.p, dncc);
  hipLaunchKernelGGL(k_scatter_alive, dim3((unsigned)nb), dim3(CT_THREADS), 0, s, fa, ncc, nb > 1 ? c->bcount.p : nullptr, ao,
                     nullptr, c->cnt + C_SURV, dncc);
}

// the kept survivors' ranks in kidx, their number in C_KEPT
static void compact_kept(chz_ctx *c, long long n, const unsigned long long *nd, hipStream_t s) {
  if (n == 0) return;
  const long long nb = (n + CT_TILE - 1) / CT_TILE;
  const FlagKept fk{c->kept.p};
  if (nb == 1) {
    hipLaunchKernelGGL(k_compact_one<FlagKept>, dim3(1), dim3(CT_THREADS), 0, s, fk, n, c->kidx.p, c->cnt + C_KEPT, nd);
    return;
  }
  hipLaunchKernelGGL(k_flag_count<FlagKept>, dim3((unsigned)nb), dim3(CT_THREADS), 0, s, fk, n, c->bcount.p, nd);
  if (nb <= CT_DIRECT) {
    hipLaunchKernelGGL(k_scatter_idx<FlagKept>, dim3((unsigned)nb), dim3(CT_THREADS), 0, s, fk, n, c->bcount.p, c->kidx.p, nd,
                       c->cnt + C_KEPT);
    return;
  }
  hipLaunchKernelGGL(k_scan_one_block, dim3(1), dim3(1024), 0, s, c->bcount.p, nb);
  hipLaunchKernelGGL(k_scatter_idx<FlagKept>, dim3((unsigned)nb), dim3(CT_THREADS), 0, s, fk, n, c->bcount.p, c->kidx.p, nd,
                     nullptr);
  hipLaunchKernelGGL(k_add_total, dim3(1), dim3(64), 0, s, c->cnt + C_KEPT, c->bcount.p + nb);
}

// bytes of the level control block for ns slots (its layout is the pinned staging area's)
static size_t ctl_in_bytes(int ns) { return counter_words(ns) * 8 + (size_t)ns * 4 + (size_t)ns; }

// the counters read back (hc: counter_words), their stripes summed into hc's stage counts and the first slot stripe
static void fold_counters(unsigned long long *hc, int ns) {
  static const int at[SG_N - 1] = {C_EVAL, C_PRE, C_NEEDT, C_CHEAP, C_CUTS, C_KEYS, C_TPASS};
  for (int i = 0; i < SG_N - 1; i++) {
    hc[at[i]] = 0;
    for (int j = 0; j < NSTRIPE; j++) hc[at[i]] += hc[C_N + j * SG_N + i];
  }
  unsigned long long *ic = hc + C_N + NSTRIPE * SG_N;
  for (int j = 1; j < slot_stripes(ns); j++)
    for (size_t x = 0; x < (size_t)ns * IC_N; x++) {
      const unsigned long long v = ic[(size_t)j * ns * IC_N + x];
      if (x % IC_N == IC_FIRST) ic[x] = std::min(ic[x], v);
      else ic[x] += v;
    }
}

// per-slot device arrays sized for `need` instance slots
static void reserve_slots(chz_ctx *c, int need) {
  if (need <= c->nslots) return;
  int ns = std::max(16, c->nslots);
  while (ns < need) ns *= 2;
  c->ctl.need((ctl_in_bytes(ns) + 7) / 8);
  c->cnt = c->ctl.p;
  c->stage = c->cnt + C_N;
  c->icnt = c->stage + NSTRIPE * SG_N;
  c->slo = (long long *)(c->cnt + bounds_at(ns));
  c->shi = c->slo + ns;
  c->d_rem = (int *)(c->cnt + counter_words(ns));
  c->d_keepi = (uint8_t *)(c->d_rem + ns);
  c->gflag.need(ns);
  HIPCHK(hipMemsetAsync(c->gflag.p, 0, (size_t)ns * 4, c->stream));   // fresh slots: no goal child known
  c->nslots = ns;
}

// the nodes [lo, hi) of every slot in a frontier of n nodes (contiguous per slot; a slot without nodes keeps the zeros of
// the level's control upload)
__global__ void k_slot_bounds(const uint32_t *inst, long long n, const unsigned long long *nd, long long *lo, long long *hi) {
  n = dev_n(n, nd);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    const uint32_t s = inst[i];
    if (i == 0 || inst[i - 1] != s) lo[s] = i;
    if (i == n - 1 || inst[i + 1] != s) hi[s] = i + 1;
  }
}

// admitted roots from the host's memory into the frontier behind its first `at` nodes
struct RootArgs {
  const int4 *u;             // nr matrices of E entries
  const int *k, *slot;
  long long nr, at;
  int4 *res;
  int *pk;
  uint8_t *g1, *g2, *tg;
  uint32_t *finst, *pb, *tp;
  uint64_t *tm;              // or null
  uint32_t *gflag;           // goal flags of ns slots to clear (a frontier of roots only), or null
  int ns;
};
template <int E> __global__ void k_put_roots(RootArgs a) {
  const long long i0 = (long long)blockIdx.x * blockDim.x + threadIdx.x, stride = (long long)gridDim.x * blockDim.x;
  for (long long i = i0; i < a.nr * E; i += stride) a.res[a.at * E + i] = a.u[i];
  for (long long i = i0; i < a.nr; i += stride) {
    const long long x = a.at + i;
    a.pk[x] = a.k[i];
    a.g1[x] = a.g2[x] = a.tg[x] = 255;
    a.finst[x] = (uint32_t)a.slot[i];
    a.pb[x] = BW_TUNK;
    a.tp[x] = NO_PARENT;
    if (a.tm) a.tm[x] = 0;
  }
  if (a.gflag)
    for (long long i = i0; i < a.ns; i += stride) a.gflag[i] = 0u;
}

// the next frontier: `distinct` gathered children (already in buffer nxt) followed by the admitted roots, which one kernel
// reads from host memory (eight copies and a synchronisation took longer than a small search's first two levels; what the
// kernel reads is written again only after the level's synchronisation)
template <int NQ> static void append_roots(chz_ctx *c, int nxt, long long distinct, uint32_t *tp, uint8_t *tg) {
  constexpr int E = 1 << (2 * NQ);
  const long long nr = (long long)c->pending.size();
  if (!nr) return;
  int4 *u = (int4 *)c->pin_io.need((size_t)nr * (E * sizeof(int4) + 8));
  int *k = (int *)(u + nr * E), *slot = k + nr;
  for (long long i = 0; i < nr; i++) {
    const Pending &q = c->pending[i];
    std::copy(q.U.begin(), q.U.end(), u + i * E);
    k[i] = q.k;
    slot[i] = c->binst[q.inst].slot;
  }
  const RootArgs ra{u, k, slot, nr, distinct, c->res[nxt].p, c->pk[nxt].p, c->g1[nxt].p, c->g2[nxt].p, tg,
                    c->finst[nxt].p, c->pb[nxt].p, tp, c->tcols ? c->tm[nxt].p : nullptr,
                    c->m ? nullptr : c->gflag.p, c->nslots};
  hipLaunchKernelGGL(k_put_roots<E>, dim3(grid_for(nr * E / 64 + 1, 1024)), dim3(256), 0, c->stream, ra);
  HIPCHK(hipGetLastError());
  for (long long i = 0; i < nr; i++) {
    c->binst[c->pending[i].inst].root_step = c->gstep + 1;
    c->forder.push_back(c->pending[i].inst);
  }
  c->pending.clear();
}

// The lexicographically first circuit of FOUND children: the child's gate, then the tree walked up to the root, one
// thread a search, WALK levels a launch (a copy and a synchronisation for every step of a walk took 0.3 ms for 12 gates)
constexpr int WALK = 32, WALK_MAX = 64;
struct WalkState { uint32_t i; int n, done; uint8_t g[WALK_MAX + 4]; };
struct WalkArgs {
  const uint32_t *par[WALK];     // levels from the highest down
  const uint8_t *gate[WALK];
  int levels, n;
  WalkState *w;                  // host memory
};
__global__ void k_walk(WalkArgs a) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= a.n || a.w[q].done) return;
  uint32_t i = a.w[q].i;
  int n = a.w[q].n, done = 0;
  for (int s = 0; s < a.levels && !done; s++) {
    const uint32_t par = a.par[s][i];
    const uint8_t g = a.gate[s][i];
    if (par == NO_PARENT) done = 1;
    else {
      if (g != CARRY_GATE && n < WALK_MAX) a.w[q].g[n++] = g;     // else a level the search waited through
      i = par;
    }
  }
  a.w[q].i = i;
  a.w[q].n = n;
  a.w[q].done = done;
}
// at[j]: FOUND child of the instance from[j]
static void walk_circuits(chz_ctx *c, const std::vector<unsigned long long> &at, const std::vector<int> &from, int G,
                          std::vector<std::vector<int>> &seq) {
  const int n = (int)at.size();
  seq.assign(n, {});
  if (!n) return;
  WalkState *w = (WalkState *)c->pin_io.need((size_t)n * sizeof(WalkState));
  int lo = c->gstep;
  for (int q = 0; q < n; q++) {
    w[q].i = (uint32_t)(at[q] / G);
    w[q].n = 1;
    w[q].done = 0;
    w[q].g[0] = (uint8_t)(at[q] % G);
    lo = std::min(lo, c->binst[from[q]].root_step);
  }
  for (int s = c->gstep; s >= lo; s -= WALK) {
    WalkArgs a{};
    a.n = n;
    a.w = w;
    for (a.levels = 0; a.levels < WALK && s - a.levels >= lo; a.levels++) {
      a.par[a.levels] = c->tree_par[s - a.levels];
      a.gate[a.levels] = c->tree_gate[s - a.levels];
    }
    hipLaunchKernelGGL(k_walk, dim3((n + 63) / 64), dim3(64), 0, c->stream, a);
  }
  HIPCHK(hipGetLastError());
  HIPCHK(hipStreamSynchronize(c->stream));
  for (int q = 0; q < n; q++) {
    seq[q].assign(w[q].g, w[q].g + w[q].n);
    std::reverse(seq[q].begin(), seq[q].end());
  }
}

static void form_columns(chz_ctx *c);

// tree levels no live search can reach any more
static void prune_tree(chz_ctx *c) {
  int oldest = c->gstep;
  for (const BInst &b : c->binst) if (b.live) oldest = std::min(oldest, b.root_step);
  for (int s = 0; s < oldest && s < (int)c->tree_par.size(); s++) {
    if (c->tree_par[s]) { c->tree_free.push_back(c->tree_par[s]); c->tree_par[s] = nullptr; }
    c->tree_gate[s] = nullptr;
  }
}

// Whether the expansion of this frontier's next level may run as the specialised kernel: the spec is one of its kind
// (std_spec), and by the searches' own roots no parent's coefficients reach 2^28 or the limit of an overflowing child (a
// sum of two terms at most doubles them), nor any child's exponent the T bound's 16 bits
static bool std_level(const chz_ctx *c) {
  if (!c->std_spec) return false;
  for (const BInst &b : c->binst) {
    if (!b.live) continue;
    const int room = b.t + 1;                     // gates from the root to this level's children
    if (room > 24 || ((uint64_t)b.coef << room) >= std::min<uint64_t>(1u << 28, c->ks.maglim)) return false;
    // a parent's exponent exceeds the root's by at most a gate's own each; alive, it is within the budget left
    const int kp = std::min(b.k + b.t * c->max_ik, b.t ? b.depth - b.t : b.k);
    if (c->ks.n + kp + c->max_ik > 16) return false;
  }
  return true;
}
// Lane groups per parent up to which this frontier's children are settled from their parents' bounds: none beside a root that
// sqrt2 divides
static int pre_split(const chz_ctx *c) {
  for (const BInst &b : c->binst) if (b.live && b.t == 0 && b.reducible) return 0;
  return PRE_SPLIT;
}
template <int NQ> static void launch_level(chz_ctx *c, int var, bool spec, dim3 grid, hipStream_t s, const ExpandArgs &ea, long long m) {
  const KSpec &ks = c->ks;
  if constexpr (NQ > 1)
    if (spec) {
      switch (var) {
        case 0: hipLaunchKernelGGL((k_level<NQ, 4, true>), grid, dim3(256), 0, s, ks, ea, m); return;
        case 2: hipLaunchKernelGGL((k_level<NQ, 6, true>), grid, dim3(256), 0, s, ks, ea, m); return;
        default: hipLaunchKernelGGL((k_level<NQ, 5, true>), grid, dim3(256), 0, s, ks, ea, m); return;
      }
    }
  switch (var) {
    case 0: hipLaunchKernelGGL((k_level<NQ, 4, false>), grid, dim3(256), 0, s, ks, ea, m); break;
    case 2: hipLaunchKernelGGL((k_level<NQ, 6, false>), grid, dim3(256), 0, s, ks, ea, m); break;
    default: hipLaunchKernelGGL((k_level<NQ, 5, false>), grid, dim3(256), 0, s, ks, ea, m); break;
  }
}

// A level of one chunk from its expansion's statuses to the kept survivors' ranks without the host: survivors, sort, exact
// dedupe, kept ranks, launched for ncc children (dncc: their number on the device) and reading the sizes that come out
// on the way from the counters.  The buffers hold ncc entries.
template <int NQ>
static void level_tail(chz_ctx *c, int cur, long long ncc, const unsigned long long *dncc, uint32_t *gflag, bool timed,
                       hipStream_t s) {
  const unsigned long long *nd = c->cnt + C_SURV;
  const uint32_t *pinst = c->finst[cur].p;
  const AliveOut ao{c->keys.p, c->info.p, 0, c->surv_o.p, c->surv_key.p, c->surv_bw.p};
  auto begin = [&](int fam) { if (timed) c->ev.begin(fam, s); };
  auto end = [&]() { if (timed) c->ev.end(s); };
  begin(K_COMPACT);
  compact_alive(c, FlagAlive{c->status.p}, ncc, ao, dncc, s);
  end();
  begin(K_SORT);
  sort_survivors(c, ncc, nd, s);
  end();
  begin(K_DEDUPE);
  const ActiveArgs aa{c->icnt, slot_stripes(c->nslots), c->nslots, c->ks.G, c->surv_o.p, pinst};
  hipLaunchKernelGGL(k_fill_kept, dim3(grid_for(ncc / 256 + 1, 256)), dim3(256), 0, s, c->kept.p, ncc, nd, aa, gflag);
  const DedupeArgs da{c->sk[0].p, c->sv[0].p, ncc, c->surv_o.p, c->surv_key.p, c->surv_bw.p, c->res[cur].p,
                      c->pk[cur].p, c->kept.p, c->cnt, pinst, nd};
  hipLaunchKernelGGL(k_dedupe_runs<NQ>, dim3(grid_for(ncc / 16 + 1, 2048)), dim3(256), 0, s, c->ks, da);
  end();
  begin(K_COMPACT);
  compact_kept(c, ncc, nd, s);
  end();
}

// the buffers of level_tail and of a gather behind it for ncc children, and the tree level of mx nodes
template <int NQ>
static void level_room(chz_ctx *c, int nxt, long long ncc, long long mx, uint32_t *&tp, uint8_t *&tg) {
  constexpr int E = 1 << (2 * NQ);
  const long long nbA = (ncc + CT_TILE - 1) / CT_TILE, nbS = (ncc + RS_TILE - 1) / RS_TILE;
  c->status.need(ncc); c->keys.need(ncc); c->info.need(ncc);
  c->bcount.need(nbA + 1);
  c->surv_o.need(ncc); c->surv_key.need(ncc); c->surv_bw.need(ncc);
  c->kept.need(ncc); c->kidx.need(ncc);
  for (int b = 0; b < 2; b++) { c->sk[b].need(ncc); c->sv[b].need(ncc); }
  c->hist.need((size_t)nbS * 256 + 1);
  c->scan_tmp.need((size_t)nbS * 256 / SC_TILE + 4);
  c->res[nxt].need((size_t)mx * E); c->pk[nxt].need(mx); c->g1[nxt].need(mx); c->g2[nxt].need(mx);
  c->pb[nxt].need(mx); c->finst[nxt].need(mx);
  if (c->tcols) c->tm[nxt].need(mx);
  tree_alloc(c, mx, tp, tg);
}

// Captured level step for levels of at most STEP_CAP parents: expansion, survivor compaction, radix sort, exact
// dedupe, the searches' continue flags and the kept compaction, in one graph built once per frontier parity with
// launches sized for the capacity; every kernel reads the level's sizes from the counters the host uploads
// (C_M, C_NCC) and those the step produces (C_SURV, C_KEPT).  The graph holds no memset node.  It
// is rebuilt when a buffer address, the slot count or the schedule it was captured with changes.  The gather runs
// after it as an ordinary launch (its tree level differs every step), then the level synchronises once.
constexpr long long STEP_CAP = 1024;
// Captures run while other threads (the request server's other engines) keep working on the device.  None of
// them may synchronise the whole device or allocate during a capture (a device-wide synchronisation includes the
// stream under capture; HIP's hipFree synchronises the device): buffer growth waits for the context's own stream
// only, and allocations, frees, device-wide synchronisations and memory queries take capture_mu, which the capture
// holds.
// Captured steps are used by batches that have held more than one search at once (the request server's engines):
// measured on MI355X, a single search runs its small levels faster as direct launches (on a reused context, Toffoli
// budget 9: 0.86 ms against 1.00 ms with captured steps, budget 12: 8.34 ms against 8.44 ms), while in the server
// they lower the latency tail.
constexpr bool kStepGraphs = true;
// Levels launched for all their children at once (below): their next frontier's room, E entries a child, is bounded by
// this many bytes (64K children of 3 qubits, 256K of 2)
constexpr long long ONCE_BYTES = 64ll << 20;
// Which frontiers k_tcols looks at: below some ten thousand nodes the expansion is as long as its longest chain, T bounds or
// not, and searches with few gates left have few T bounds to save (24 searches of up to 10 gates in a batch, with every
// frontier of 4K nodes looked at: 9.57 -> 10.05 ms; of 32K, and 6 gates left: 9.6)
constexpr long long TCOLS_MIN = 32768;
constexpr int TCOLS_LEFT = 6;
constexpr int STEP_BUCKET = 10;    // the schedule of the 1,024-parent bucket drives the captured expansion

template <int NQ>
static void step_graph(chz_ctx *c, int cur, long long m, const unsigned long long *hc_in, unsigned long long *hc,
                       uint32_t *&tp, uint8_t *&tg) {
  constexpr int N = 1 << NQ, E = N * N, CPW = 64 / E;
  (void)N;
  const KSpec &ks = c->ks;
  const int G = ks.G, nxt = cur ^ 1, ns = c->nslots;
  const long long cap = STEP_CAP, ncap = cap * G;
  const long long mx = ncap + (long long)c->pending.size();
  level_room<NQ>(c, nxt, ncap, mx, tp, tg);
  const chz_ctx::Sched sc = c->sched[STEP_BUCKET];
  const bool spec = std_level(c);
  const int psplit = pre_split(c);
  const uint32_t *pinst = c->finst[cur].p;
  const std::vector<uintptr_t> key = {
      (uintptr_t)c->res[cur].p, (uintptr_t)c->pk[cur].p, (uintptr_t)c->g1[cur].p, (uintptr_t)c->g2[cur].p,
      (uintptr_t)c->pb[cur].p, (uintptr_t)c->tm[cur].p, (uintptr_t)pinst, (uintptr_t)c->status.p, (uintptr_t)c->keys.p, (uintptr_t)c->info.p,
      (uintptr_t)c->cnt, (uintptr_t)c->d_rem, (uintptr_t)c->d_keepi, (uintptr_t)c->icnt,
      (uintptr_t)c->bcount.p, (uintptr_t)c->surv_o.p, (uintptr_t)c->surv_key.p, (uintptr_t)c->surv_bw.p,
      (uintptr_t)c->kept.p, (uintptr_t)c->kidx.p, (uintptr_t)c->sk[0].p, (uintptr_t)c->sk[1].p,
      (uintptr_t)c->sv[0].p, (uintptr_t)c->sv[1].p, (uintptr_t)c->hist.p, (uintptr_t)c->scan_tmp.p,
      (uintptr_t)c->gflag.p, (uintptr_t)ns, (uintptr_t)sc.var, (uintptr_t)sc.cap,
      (uintptr_t)sc.tw, (uintptr_t)spec, (uintptr_t)psplit};
  chz_ctx::StepGraph &sg = c->sgraph[cur];
  if (!sg.exec || sg.key != key) {
    if (sg.exec) { HIPCHK(hipGraphExecDestroy(sg.exec)); sg.exec = nullptr; }
    const unsigned long long *dm = c->cnt + C_M, *dncc = c->cnt + C_NCC;
    hipStream_t s = c->stream;
    hipGraph_t graph = nullptr;
    // no device-wide or allocating HIP call from another thread while this stream is captured (capture_mu)
    std::lock_guard<std::recursive_mutex> capture_lock(capture_mu());
    HIPCHK(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
    ExpandArgs ea{c->res[cur].p, c->pk[cur].p, c->g1[cur].p, c->g2[cur].p, 0,
                  c->status.p, c->keys.p, c->info.p, c->pb[cur].p, c->tm[cur].p, c->stage, pinst, c->d_rem, c->d_keepi,
                  c->icnt, slot_stripes(ns), ns * IC_N, 1, dm, sc.tw, psplit, c->goal_skip ? c->gflag.p : nullptr};
    const dim3 grid(grid_for((cap * G + CPW - 1) / CPW, sc.cap));
    launch_level<NQ>(c, sc.var, spec, grid, s, ea, cap);
    level_tail<NQ>(c, cur, ncap, dncc, nullptr, false, s);
    hipError_t e = hipGetLastError();
    const hipError_t ec = hipStreamEndCapture(s, &graph);
    if (e == hipSuccess) e = ec;
    if (e == hipSuccess) e = hipGraphInstantiate(&sg.exec, graph, nullptr, nullptr, 0);
    if (graph) (void)hipGraphDestroy(graph);
    if (e != hipSuccess) {
      sg.exec = nullptr;
      set_err(std::string("HIP error: ") + hipGetErrorString(e) + " while capturing a level step");
      throw DeviceError();
    }
    sg.key = key;
  }
  HIPCHK(hipMemcpyAsync(c->cnt, hc_in, C_N * 8, hipMemcpyHostToDevice, c->stream));
  c->ev.begin(K_STEP, c->stream);
  HIPCHK(hipGraphLaunch(sg.exec, c->stream));
  c->ev.end(c->stream);
  const GatherArgs ga{c->kidx.p, ncap, c->surv_o.p, c->res[cur].p, c->pk[cur].p, c->g1[cur].p,
                      c->res[nxt].p, c->pk[nxt].p, c->g1[nxt].p, c->g2[nxt].p, tp, tg, pinst, c->finst[nxt].p,
                      c->surv_bw.p, c->pb[nxt].p, c->cnt + C_KEPT, c->goal_skip ? c->gflag.p : nullptr, CPW};
  HIPCHK(hipMemsetAsync(c->gflag.p, 0, (size_t)ns * 4, c->stream));   // the graph's expansion has read them
  c->ev.begin(K_GATHER, c->stream);
  hipLaunchKernelGGL(k_gather<NQ>, dim3(grid_for((ncap + CPW - 1) / CPW)), dim3(256), 0, c->stream, ks, ga, c->pb[cur].p, c->cols_on ? c->tm[cur].p : nullptr, c->tcols ? c->tm[nxt].p : nullptr);
  c->ev.end(c->stream);
  HIPCHK(hipMemcpyAsync(hc, c->cnt, counter_words(ns) * 8, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  // what a large level before this one outgrew; the few megabytes that small levels outgrow wait for the next large one, since
  // giving blocks back waits for a capture that another engine has open
  size_t held = 0;
  for (const auto &b : c->retired) held += b.second;
  if (held > (size_t)ONCE_BYTES) settle(c->retired);
  fold_counters(hc, ns);
  c->ev.flush(c->k_ms, c->k_launch);
  if (hc[C_REPOVF]) { set_err("a dedupe run holds more distinct classes than its buffer"); throw DeviceError(); }
  c->k_work[K_GATHER] += (double)hc[C_KEPT] * (E * 16.0 * 2.0 + 16.0);
}

// One level of every live search of the batch (src/cheese.cu:1249-1377 per search): expansion in chunks,
// survivor compaction, sort, exact dedupe, next frontier; then the searches admitted since the last step join
// the new frontier as roots.  Level lines and results go to the context's event queue.
template <int NQ> static void batch_step(chz_ctx *c) {
  constexpr int N = 1 << NQ, E = N * N, CPW = 64 / E;
  const KSpec &ks = c->ks;
  const int G = ks.G;
  if (c->m == 0 && c->pending.empty()) return;
  if (c->m == 0) {   // a frontier of roots only
    c->cols_on = false;
    const long long nr = (long long)c->pending.size();
    const int nxt = c->cur ^ 1;
    c->res[nxt].need(nr * E); c->pk[nxt].need(nr); c->g1[nxt].need(nr); c->g2[nxt].need(nr); c->finst[nxt].need(nr);
    c->pb[nxt].need(nr);
    if (c->tcols) c->tm[nxt].need(nr);
    uint32_t *tp = nullptr;
    uint8_t *tg = nullptr;
    tree_alloc(c, nr, tp, tg);
    c->tree_par.push_back(tp);
    c->tree_gate.push_back(tg);
    c->gstep = (int)c->tree_par.size() - 1;
    c->gstep--;                 // append_roots marks roots with gstep + 1
    append_roots<NQ>(c, nxt, 0, tp, tg);
    c->gstep++;
    c->cur = nxt;
    c->m = nr;
    for (BInst &b : c->binst) if (b.live) b.nodes = 1;
  }
  const double tl = now_s();
  const int cur = c->cur;
  const long long m = c->m;
  // per-level memory planning: the searches expanded this step are the longest prefix of the frontier (whole
  // searches, in frontier order, at least one) whose planned bytes fit the budget beside the frontier held: per
  // parent its children's records and its share of the next frontier, by the search's last growth (a prior of
  // kGrowthPrior before its first level); the others wait a step, carried unexpanded
  long long ma = m;
  std::vector<char> carried(c->binst.size(), 0);
  if (c->mem_budget > 0 && m > 0) {
    constexpr double node_b = E * 16.0 + 24.0, child_b = 48.0, kGrowthPrior = 8.0;
    const double held = (double)m * node_b;
    double plan = 0;
    long long acc = 0;
    bool stop = false;
    for (int bi : c->forder) {
      const BInst &b = c->binst[bi];
      if (!b.live) continue;
      const double g = std::min<double>(G, b.growth > 0 ? b.growth : kGrowthPrior);
      const double need = (double)b.nodes * (G * child_b + g * node_b);
      if (acc > 0 && (stop || held + plan + need > c->mem_budget)) { stop = true; carried[bi] = 1; continue; }
      plan += need;
      acc += b.nodes;
    }
    ma = acc;
  }
  // the level's control block staged in pinned memory with the device block's layout, uploaded in one copy:
  // [counters in | per-slot counters in | rem | keepi], then [counters out | per-slot counters out] (read back
  // in one copy), the kept total and the per-slot active flags
  const int ns = c->nslots;
  const size_t in_bytes = ctl_in_bytes(ns), o_out = (in_bytes + 63) & ~(size_t)63,
               o_act = o_out + counter_words(ns) * 8;
  uint8_t *pin = c->pin.need(o_act + ns);
  unsigned long long *hc_in = (unsigned long long *)pin, *ic_in = hc_in + C_N + NSTRIPE * SG_N;
  unsigned long long *hc = (unsigned long long *)(pin + o_out), *ic = hc + C_N + NSTRIPE * SG_N;
  int *rem = (int *)(hc_in + counter_words(ns));
  uint8_t *keepi = (uint8_t *)(rem + ns), *active = pin + o_act;
  std::memset(hc_in, 0, counter_words(ns) * 8);
  for (int s = 0; s < ns; s++) {
    rem[s] = 0;
    keepi[s] = active[s] = 0;
    for (int j = 0; j < slot_stripes(ns); j++) ic_in[((size_t)j * ns + s) * IC_N + IC_FIRST] = ~0ull;
  }
  for (const BInst &b : c->binst)
    if (b.live) { rem[b.slot] = b.depth - (b.t + 1); keepi[b.slot] = b.t + 1 < b.depth; }
  HIPCHK(hipMemcpyAsync(c->ctl.p, pin, in_bytes, hipMemcpyHostToDevice, c->stream));
  const long long chunk = c->opts.chunk > 0 ? c->opts.chunk : (1ll << 20);
  const uint32_t *pinst = c->finst[cur].p;
  const int nxt = cur ^ 1;
  long long nsurv = 0, distinct = 0;
  bool gflag_clear = false;          // the goal flags were cleared by this level's kept fill
  bool once = false, counted = false;
  uint32_t *tp = nullptr;
  uint8_t *tg = nullptr;
  // small levels run as one captured graph (expansion through kept compaction) plus the gather: one
  // synchronisation per level instead of two, and one launch instead of about twenty
  const bool graphed = kStepGraphs && c->shared_steps && !c->tuning && !c->gt_filter && c->opts.dedupe && m > 0 &&
                       m <= STEP_CAP && m <= chunk && ma == m;
  if (graphed) {
    for (int i = 0; i < C_N; i++) hc_in[i] = 0;
    hc_in[C_M] = (unsigned long long)m;
    hc_in[C_NCC] = (unsigned long long)(m * G);
    step_graph<NQ>(c, cur, m, hc_in, hc, tp, tg);
    nsurv = (long long)hc[C_SURV];
    distinct = (long long)hc[C_KEPT];
    c->k_work[K_STEP] += expand_ops(c, NQ, hc) + (double)(m * G) + (double)nsurv * (24.0 + 16.0 + 4 * 20.0 + 9.0);
    static const int stage_ctr[6] = {C_EVAL, C_CHEAP, C_CUTS, C_NEEDT, C_KEYS, C_TPASS};
    for (int i = 0; i < 6; i++) c->k_stage[i] += (double)hc[stage_ctr[i]];
    for (const BInst &b : c->binst)
      if (b.live) {
        const unsigned long long *x = &ic[(size_t)b.slot * IC_N];
        active[b.slot] = !x[IC_FOUND] && !x[IC_OVF] && keepi[b.slot];
      }
  } else {
  const bool alone = c->pending.empty() && chz_batch_live(c) == 1;
  // levels of few children need the host for nothing between their expansion and the next frontier: launched for all
  // children of the level, with one synchronisation and one copy at the end
  once = !c->tuning && !c->gt_filter && c->opts.dedupe && c->pending.empty() && ma == m && ma <= chunk && ma * G * E * 16 <= ONCE_BYTES;
  const long long maxcc = std::min<long long>(chunk, std::max<long long>(ma, 1)) * G;
  const bool spec = std_level(c);
  if (once) level_room<NQ>(c, nxt, maxcc, maxcc, tp, tg);

  c->status.need(maxcc);
  c->info.need(maxcc);
  c->keys.need(maxcc);
  c->bcount.need((maxcc + CT_TILE - 1) / CT_TILE + 1);
  // survivors of every chunk append at the device-side count C_SURV: the buffers hold every child of the level
  c->surv_o.need((size_t)std::max<long long>(ma, 1) * G);
  c->surv_key.need((size_t)std::max<long long>(ma, 1) * G);
  c->surv_bw.need((size_t)std::max<long long>(ma, 1) * G);
  for (long long off = 0; off < ma; off += chunk) {
    const long long cm = std::min(chunk, ma - off), ncc = cm * G;
    // the schedule of this chunk's size bucket: few parents split each parent's candidates over several lane
    // groups so the level fills the GPU
    const int bucket = std::min(31, 63 - __builtin_clzll((unsigned long long)cm));
    const chz_ctx::Sched sc = c->tuning ? c->force : c->sched[bucket];
    const int gsplit = (int)std::max<long long>(1, std::min<long long>(G, ((long long)sc.tw * CPW + cm - 1) / cm));
    ExpandArgs ea{c->res[cur].p, c->pk[cur].p, c->g1[cur].p, c->g2[cur].p, off,
                  c->status.p, c->keys.p, c->info.p, c->pb[cur].p, c->tm[cur].p, c->stage, pinst, c->d_rem, c->d_keepi,
                  c->icnt, slot_stripes(ns), ns * IC_N, gsplit, nullptr, 0, pre_split(c), c->goal_skip ? c->gflag.p : nullptr};
    const dim3 grid(grid_for((cm * gsplit + CPW - 1) / CPW, sc.cap));
    hipEvent_t te0 = nullptr, te1 = nullptr;
    if (c->tuning) {
      te0 = c->ev.take();
      te1 = c->ev.take();
      HIPCHK(hipEventRecord(te0, c->stream));
    }
    c->ev.begin(K_EXPAND, c->stream);
    launch_level<NQ>(c, sc.var, spec, grid, c->stream, ea, cm);
    c->ev.end(c->stream);
    if (c->tuning) {
      HIPCHK(hipEventRecord(te1, c->stream));
      c->tune_ev.push_back({bucket, {te0, te1}});
    }
    const long long nb = (ncc + CT_TILE - 1) / CT_TILE;
    if (once || ncc == 0) break;
    const FlagAlive fa{c->status.p};
    const AliveOut ao{c->keys.p, c->info.p, off * G, c->surv_o.p, c->surv_key.p, c->surv_bw.p};
    c->ev.begin(K_COMPACT, c->stream);
    if (ncc <= CT_DIRECT * CT_TILE && ma <= chunk) compact_alive(c, fa, ncc, ao, nullptr, c->stream);
    else {
      hipLaunchKernelGGL(k_flag_count<FlagAlive>, dim3((unsigned)nb), dim3(CT_THREADS), 0, c->stream, fa, ncc,
                         c->bcount.p);
      hipLaunchKernelGGL(k_scan_one_block, dim3(1), dim3(1024), 0, c->stream, c->bcount.p, nb);
      hipLaunchKernelGGL(k_scatter_alive, dim3((unsigned)nb), dim3(CT_THREADS), 0, c->stream, fa, ncc, c->bcount.p, ao,
                         c->cnt + C_SURV, nullptr, nullptr);
      hipLaunchKernelGGL(k_add_total, dim3(1), dim3(64), 0, c->stream, c->cnt + C_SURV, c->bcount.p + nb);
    }
    c->ev.end(c->stream);
    c->k_work[K_COMPACT] += (double)ncc;
  }
  if (once) {
    level_tail<NQ>(c, cur, maxcc, nullptr, c->gflag.p, true, c->stream);
    gflag_clear = true;
    const GatherArgs ga{c->kidx.p, maxcc, c->surv_o.p, c->res[cur].p, c->pk[cur].p, c->g1[cur].p,
                        c->res[nxt].p, c->pk[nxt].p, c->g1[nxt].p, c->g2[nxt].p, tp, tg, pinst, c->finst[nxt].p,
                        c->surv_bw.p, c->pb[nxt].p, c->cnt + C_KEPT, c->goal_skip ? c->gflag.p : nullptr, CPW};
    c->ev.begin(K_GATHER, c->stream);
    hipLaunchKernelGGL(k_gather<NQ>, dim3(grid_for((maxcc / 4 + CPW - 1) / CPW)), dim3(256), 0, c->stream, ks, ga, c->pb[cur].p, c->cols_on ? c->tm[cur].p : nullptr, c->tcols ? c->tm[nxt].p : nullptr);
    c->ev.end(c->stream);
    if (!alone) {
      hipLaunchKernelGGL(k_slot_bounds, dim3(grid_for(maxcc / 256 + 1, 256)), dim3(256), 0, c->stream, c->finst[nxt].p, maxcc,
                         c->cnt + C_KEPT, c->slo, c->shi);
      counted = true;
    }
  }
  HIPCHK(hipMemcpyAsync(hc, c->cnt, counter_words(ns) * 8, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(hipStreamSynchronize(c->stream));
  fold_counters(hc, ns);
  c->ev.flush(c->k_ms, c->k_launch);
  nsurv = (long long)hc[C_SURV];
  c->k_work[K_COMPACT] += (double)nsurv * 24.0;
  c->k_work[K_EXPAND] += expand_ops(c, NQ, hc);
  static const int stage_ctr[6] = {C_EVAL, C_CHEAP, C_CUTS, C_NEEDT, C_KEYS, C_TPASS};
  for (int i = 0; i < 6; i++) c->k_stage[i] += (double)hc[stage_ctr[i]];
  // searches that end at this level with a circuit or an overflow; the rest continue if their budget allows
  for (const BInst &b : c->binst)
    if (b.live) {
      const unsigned long long *x = &ic[(size_t)b.slot * IC_N];
      active[b.slot] = !x[IC_FOUND] && !x[IC_OVF] && keepi[b.slot];
    }
  settle(c->retired);
  if (once) {
    if (hc[C_REPOVF]) { set_err("a dedupe run holds more distinct classes than its buffer"); throw DeviceError(); }
    distinct = (long long)hc[C_KEPT];
    c->k_work[K_COMPACT] += (double)(m * G);
    c->k_work[K_SORT] += (double)nsurv * (16.0 + 4 * (4.0 + 16.0));
    c->k_work[K_DEDUPE] += (double)nsurv * 9.0;
    c->k_work[K_GATHER] += (double)distinct * (E * 16.0 * 2.0 + 16.0);
  } else if (nsurv > 0) {
    c->kept.need(nsurv);
    c->kidx.need(nsurv);
    const ActiveArgs aa{c->icnt, slot_stripes(ns), ns, G, c->surv_o.p, pinst};
    gflag_clear = true;
    if (c->opts.dedupe && nsurv > 1) {
      c->ev.begin(K_SORT, c->stream);
      sort_survivors(c, nsurv, nullptr, c->stream);
      c->ev.end(c->stream);
      c->k_work[K_SORT] += (double)nsurv * (16.0 + 4 * (4.0 + 16.0));
      c->ev.begin(K_DEDUPE, c->stream);
      hipLaunchKernelGGL(k_fill_kept, dim3(grid_for(nsurv / 256 + 1)), dim3(256), 0, c->stream, c->kept.p, nsurv,
                         nullptr, aa, c->gflag.p);
      const DedupeArgs da{c->sk[0].p, c->sv[0].p, nsurv, c->surv_o.p, c->surv_key.p, c->surv_bw.p,
                          c->res[cur].p, c->pk[cur].p, c->kept.p, c->cnt, pinst, nullptr};
      hipLaunchKernelGGL(k_dedupe_runs<NQ>, dim3(grid_for(nsurv / 4 + 1, 4096)), dim3(256), 0, c->stream, ks, da);
      c->ev.end(c->stream);
      c->k_work[K_DEDUPE] += (double)nsurv * 9.0;
    } else {
      hipLaunchKernelGGL(k_fill_kept, dim3(grid_for(nsurv / 256 + 1)), dim3(256), 0, c->stream, c->kept.p, nsurv,
                         nullptr, aa, c->gflag.p);
    }
    if (c->gt_filter)      // a table build: classes already in the table (lower levels) are dropped
      hipLaunchKernelGGL(k_gt_filter<NQ>, dim3(grid_for(nsurv / CPW + 1)), dim3(256), 0, c->stream, ks,
                         c->gt_filter->dev(), c->surv_o.p, c->surv_key.p, nsurv, c->res[cur].p, c->pk[cur].p,
                         c->kept.p);
    const long long nb = (nsurv + CT_TILE - 1) / CT_TILE;
    c->bcount.need(nb + 1);
    c->ev.begin(K_COMPACT, c->stream);
    compact_kept(c, nsurv, nullptr, c->stream);
    c->ev.end(c->stream);
    HIPCHK(hipMemcpyAsync(hc, c->cnt, C_N * 8, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(hipStreamSynchronize(c->stream));
    if (hc[C_REPOVF]) { set_err("a dedupe run holds more distinct classes than its buffer"); throw DeviceError(); }
    distinct = (long long)hc[C_KEPT];
  }
  }   // normal path
  // next frontier: kept children, then the searches admitted since the last step.  The goal flags describe the
  // frontier being expanded until here; the gather sets them for the next one.
  const bool gathered = graphed || once;      // the next frontier's children are in place
  if (!graphed && !gflag_clear) HIPCHK(hipMemsetAsync(c->gflag.p, 0, (size_t)ns * 4, c->stream));
  const long long ncarry = m - ma;            // nodes of the searches that waited
  const long long mn = distinct + ncarry + (long long)c->pending.size();
  std::vector<long long> cnts(c->nslots, 0);
  if (mn) {
    if (!gathered) {
      c->res[nxt].need((size_t)mn * E); c->pk[nxt].need(mn); c->g1[nxt].need(mn); c->g2[nxt].need(mn);
      c->pb[nxt].need(mn);
      if (c->tcols) c->tm[nxt].need(mn);
      c->finst[nxt].need(mn);
      tree_alloc(c, mn, tp, tg);
    }
    if (distinct && !gathered) {
      const GatherArgs ga{c->kidx.p, distinct, c->surv_o.p, c->res[cur].p, c->pk[cur].p, c->g1[cur].p,
                          c->res[nxt].p, c->pk[nxt].p, c->g1[nxt].p, c->g2[nxt].p, tp, tg, pinst, c->finst[nxt].p,
                          c->surv_bw.p, c->pb[nxt].p, nullptr, c->goal_skip ? c->gflag.p : nullptr,
                          gather_tile<NQ>(distinct)};
      c->ev.begin(K_GATHER, c->stream);
      hipLaunchKernelGGL(k_gather<NQ>, dim3(grid_for((distinct + ga.tn - 1) / ga.tn)), dim3(256), 0, c->stream, ks,
                         ga, c->pb[cur].p, c->cols_on ? c->tm[cur].p : nullptr, c->tcols ? c->tm[nxt].p : nullptr);
      c->ev.end(c->stream);
      c->k_work[K_GATHER] += (double)distinct * (E * 16.0 * 2.0 + 16.0);
      int left = 0;                 // the most gates a search has left after this level
      for (const BInst &b : c->binst) if (b.live) left = std::max(left, b.depth - (b.t + 1));
      if (c->tcols && distinct >= TCOLS_MIN && left >= TCOLS_LEFT) {
        form_columns(c);
        c->cols_on = true;
        hipLaunchKernelGGL(k_tcols, dim3(grid_for(distinct / 16 + 1, 4096)), dim3(256), 0, c->stream, ks, c->res[nxt].p, c->pk[nxt].p,
                           c->pb[nxt].p, c->finst[nxt].p, c->d_rem, c->goal_skip ? c->gflag.p : nullptr, c->tm[nxt].p, distinct);
      }
    }
    const bool single = c->pending.empty() && chz_batch_live(c) == 1;
    if (c->gt_filter && distinct)   // a table build keeps every level, resident, with its classes' keys
      gt_add_level<NQ>(ks, *c->gt_filter, c->res[nxt].p, c->pk[nxt].p, tp, tg, distinct, c->stream);
    if (ncarry) {                   // the waiting searches' nodes follow the gathered ones, unchanged
      HIPCHK(hipMemcpyAsync(c->res[nxt].p + (size_t)distinct * E, c->res[cur].p + (size_t)ma * E,
                            (size_t)ncarry * E * sizeof(int4), hipMemcpyDeviceToDevice, c->stream));
      HIPCHK(hipMemcpyAsync(c->pk[nxt].p + distinct, c->pk[cur].p + ma, (size_t)ncarry * 4, hipMemcpyDeviceToDevice,
                            c->stream));
      HIPCHK(hipMemcpyAsync(c->g1[nxt].p + distinct, c->g1[cur].p + ma, (size_t)ncarry, hipMemcpyDeviceToDevice,
                            c->stream));
      HIPCHK(hipMemcpyAsync(c->g2[nxt].p + distinct, c->g2[cur].p + ma, (size_t)ncarry, hipMemcpyDeviceToDevice,
                            c->stream));
      HIPCHK(hipMemcpyAsync(c->pb[nxt].p + distinct, c->pb[cur].p + ma, (size_t)ncarry * 4, hipMemcpyDeviceToDevice,
                            c->stream));
      if (c->tcols)
        HIPCHK(hipMemcpyAsync(c->tm[nxt].p + distinct, c->tm[cur].p + ma, (size_t)ncarry * 8, hipMemcpyDeviceToDevice, c->stream));
      HIPCHK(hipMemcpyAsync(c->finst[nxt].p + distinct, c->finst[cur].p + ma, (size_t)ncarry * 4,
                            hipMemcpyDeviceToDevice, c->stream));
      hipLaunchKernelGGL(k_carry_tree, dim3(grid_for(ncarry / 64 + 1)), dim3(256), 0, c->stream, tp + distinct,
                         tg + distinct, ncarry, ma);
      for (size_t bi = 0; bi < carried.size(); bi++) c->carried_levels += carried[bi];
    }
    append_roots<NQ>(c, nxt, distinct + ncarry, tp, tg);
    c->tree_par.push_back(tp);
    c->tree_gate.push_back(tg);
    if (single) {   // one search: its nodes are the whole frontier (its kernel times are read next step)
      for (const BInst &b : c->binst) if (b.live) cnts[b.slot] = mn;
    } else {
      const long long *lo = (const long long *)(hc + bounds_at(ns));
      if (!counted) {
        hipLaunchKernelGGL(k_slot_bounds, dim3(grid_for(mn / 64 + 1)), dim3(256), 0, c->stream, c->finst[nxt].p, mn, nullptr,
                           c->slo, c->shi);
        HIPCHK(hipMemcpyAsync(hc + bounds_at(ns), c->slo, (size_t)ns * 16, hipMemcpyDeviceToHost, c->stream));
        HIPCHK(hipStreamSynchronize(c->stream));
        settle(c->retired);
      }
      for (int x = 0; x < ns; x++) cnts[x] = lo[ns + x] - lo[x];
      c->ev.flush(c->k_ms, c->k_launch);
    }
  } else {
    if (gathered && tp) c->tree_free.push_back(tp);    // the level's tree block holds no node
    if (!once) HIPCHK(hipStreamSynchronize(c->stream));
    c->ev.flush(c->k_ms, c->k_launch);
  }
  // events of this level, per search
  std::vector<unsigned long long> found_at;
  std::vector<int> found_by;
  std::vector<std::vector<int>> found_seq;
  for (size_t bi = 0; bi < c->binst.size(); bi++) {
    const BInst &b = c->binst[bi];
    if (!b.live || b.root_step > c->gstep || (bi < carried.size() && carried[bi])) continue;
    const unsigned long long *x = &ic[(size_t)b.slot * IC_N];
    if (x[IC_OVF] || !x[IC_FOUND]) continue;
    found_at.push_back(x[IC_FIRST]);
    found_by.push_back((int)bi);
  }
  walk_circuits(c, found_at, found_by, G, found_seq);
  const double now = now_s();
  for (size_t bi = 0; bi < c->binst.size(); bi++) {
    BInst &b = c->binst[bi];
    if (!b.live || b.root_step > c->gstep) continue;      // admitted in this step: it has not expanded yet
    if (bi < carried.size() && carried[bi]) continue;      // waited this step: no level
    const unsigned long long *x = &ic[(size_t)b.slot * IC_N];
    chz_event evn{};
    evn.tag = b.tag;
    if (x[IC_OVF]) {
      evn.kind = 1;
      evn.result.rc = 4;
      evn.result.seconds = now - b.t0;
      set_err("residual coefficients exceed the storage type (int32)");
    } else if (x[IC_FOUND]) {
      const std::vector<int> &seq = found_seq[std::find(found_by.begin(), found_by.end(), (int)bi) - found_by.begin()];
      evn.kind = 1;
      evn.result.rc = 0;
      evn.result.len = (int)seq.size();
      evn.result.found = (long)x[IC_FOUND];
      for (size_t j = 0; j < seq.size() && j < CHZ_DMAX; j++) evn.result.circuit[j] = seq[j];
      evn.result.seconds = now - b.t0;
    } else {
      const long long dist = active[b.slot] ? cnts[b.slot] : 0;
      chz_event lv{};
      lv.tag = b.tag;
      lv.kind = 0;
      lv.level.t = b.t + 1;
      lv.level.parents = (long)b.nodes;
      lv.level.prefixes = (long)(b.nodes * G - (long long)x[IC_W2]);
      lv.level.cut_w3 = (long)x[IC_W3];
      lv.level.cut_lb = (long)x[IC_DEAD];
      lv.level.survivors = (long)x[IC_ALIVE];
      lv.level.distinct = (long)dist;
      lv.level.proved_unsat = dist ? 0 : 1;
      lv.level.seconds = now - tl;
      c->events.push_back(lv);
      b.t++;
      if (b.nodes > 0) b.growth = (double)dist / (double)b.nodes;
      b.nodes = dist;
      if (dist) continue;
      evn.kind = 1;
      evn.result.rc = 1;
      evn.result.seconds = now - b.t0;
    }
    c->events.push_back(evn);
    b.live = false;
  }
  // roots admitted in this step
  for (BInst &b : c->binst)
    if (b.live && b.root_step == c->gstep + 1) b.nodes = cnts[b.slot];
  c->cur = nxt;
  c->m = mn;
  c->gstep++;
  c->forder.erase(std::remove_if(c->forder.begin(), c->forder.end(), [&](int bi) { return !c->binst[bi].live; }),
                  c->forder.end());
  prune_tree(c);
}

// LevelTabs for a spec: the term descriptors and headers of its candidates, its symmetries' entry positions (n = 3),
// its cx table (when it fits) and the entry sources of its cut matrices
static void build_level_tabs(SpecTabs &TS, const std::vector<DevGate> &dg, const KSpec &k, const chz::SymGroup &grp,
                             const HostSpec &s) {
  std::memset(&TS, 0, sizeof TS);
  LevelTabs &T = TS.level;
  const int n = k.n, N = 1 << n, GS = N * N;
  for (int g = 0; g < k.G; g++) {
    const DevGate &d = dg[g];
    bool terms = true;
    for (int e = 0; e < GS; e++) {
      const int ec = e & (N - 1);
      int lc = (ec >> d.q[0]) & 1;
      if (d.nq > 1) lc |= ((ec >> d.q[1]) & 1) << 1;
      if (d.nq > 2) lc |= ((ec >> d.q[2]) & 1) << 2;
      const int cb = ec & ~d.mask;
      uint32_t desc = 0;
      uint32_t ring = 0;
      int nt = 0;
      for (int m = 0; d.unit && m < d.L; m++) {
        const int p = d.ph[m * d.L + lc];
        if (p < 0) continue;
        int x = cb | ((m & 1) << d.q[0]);
        if (d.nq > 1) x |= ((m >> 1) & 1) << d.q[1];
        if (d.nq > 2) x |= ((m >> 2) & 1) << d.q[2];
        if (nt < 2) {
          desc |= (uint32_t)(x | (p << 3)) << (6 * nt);
          ring |= (uint32_t)(x * RING + 3 - (p & 3) | (p >> 2 & 1) << 6) << (7 * nt);
        }
        nt++;
      }
      T.term[g * 64 + e] = (uint16_t)(ring | (nt == 2 ? 0x4000u : 0u));
      terms = terms && d.unit && nt >= 1 && nt <= 2;
      TS.sdesc[g * 64 + e] = (uint16_t)(!d.unit || nt == 0 || nt > 2 ? 0x8000u : nt == 2 ? desc | 0x1000u : desc);
    }
    int kind = 0;
    if (d.unit) {
      kind = 2;                                // permutation: one nonzero per column
      for (int lc = 0; lc < d.L; lc++) {
        int nz = 0;
        for (int m = 0; m < d.L; m++) nz += d.ph[m * d.L + lc] >= 0;
        if (nz != 1) kind = 1;
      }
    }
    const int fall = kind == 2 ? 0 : std::min(31, std::max(0, s.gates[g].gk));
    bool had = d.nq == 1 && d.unit && d.ik == 1 && s.gates[g].gk == 1;
    for (int i = 0; had && i < 4; i++) had = d.ph[i] == 0 || d.ph[i] == 4;
    T.head[g] = make_uint4((uint32_t)std::min(255, d.tdel) | (uint32_t)(d.mask & 7) << 8 | (uint32_t)fall << 11 |
                               (uint32_t)had << 16 | (uint32_t)d.cls << 24,
                           (uint32_t)d.cdel, (uint32_t)d.ik,
                           (uint32_t)terms | (uint32_t)(kind == 2) << 1 | (uint32_t)(d.cutloc & 0xffff) << 8);
  }
  if (n == 3) {
    // per order of the qubits' sums, the symmetries that make it smallest: qubit q goes to place image(q)
    for (int code = 0; code < 64; code++)
      for (int cj = 0; cj < 2; cj++) {
        int best = 1 << 30, score[16];
        for (int y = 0; y < k.nsym; y++) {
          score[y] = 0;
          for (int q = 0; q < 3; q++) {
            const int to = grp.bperm[y * 8 + (1 << q)] >> 1;      // 1, 2, 4 -> 0, 1, 2
            score[y] |= ((code >> (2 * q)) & 3) << (4 - 2 * to);
          }
          if (grp.conj[y] == cj) best = std::min(best, score[y]);
        }
        for (int y = 0; y < k.nsym; y++)
          if (grp.conj[y] == cj && score[y] == best) T.kt.adm[code] |= (uint16_t)(1u << y);
      }
    for (int y = 0; y < 16 && y < k.nsym; y++)
      for (int e = 0; e < 64; e++) T.spos[y * 64 + e] = (uint8_t)(grp.bperm[y * 8 + (e >> 3)] * 8 + grp.bperm[y * 8 + (e & 7)]);
  }
  if (k.cxlds && k.have_table)
    for (int i = 0; i < CXL_MAX && i < k.ncx; i++) T.scx[i] = (uint8_t)s.cxtable[i];
  for (int i = 0; i < CSRC_MAX * GS; i++) {
    if (i / GS >= k.ncuts) continue;
    const int le = i % GS, A = k.cutmask[i / GS], sa = k.cutsize[i / GS];
    T.scsrc[i] = (uint8_t)(n == 3 ? cut_source<3>(le, A, sa) : n == 2 ? cut_source<2>(le, A, sa) : cut_source<1>(le, A, sa));
  }
}

static void upload_spec(chz_ctx *c) {
  const HostSpec &s = c->hs;
  const int N = s.N(), G = s.G();
  std::vector<DevGate> dg(G);
  double terms = 0, columns = 0, qubits = 0;
  for (int g = 0; g < G; g++) {
    const HostGate &h = s.gates[g];
    DevGate &d = dg[g];
    std::memset(&d, 0, sizeof d);
    d.nq = h.nq;
    d.L = 1 << h.nq;
    d.ik = h.ik;
    for (int j = 0; j < h.nq; j++) { d.q[j] = h.q[j]; d.mask |= 1 << h.q[j]; }
    d.unit = 1;
    for (int i = 0; i < d.L * d.L; i++) {
      const Zq &z = h.inv[i];
      d.inv[i] = make_int4((int)z.a, (int)z.b, (int)z.c, (int)z.d);
      // +-w^p has exactly one coefficient equal to +-1: w^p for p < 4 at index p, -w^p = w^(p+4)
      const int nz = (z.a != 0) + (z.b != 0) + (z.c != 0) + (z.d != 0);
      if (!nz) { d.ph[i] = -1; continue; }
      const int64_t cf[4] = {z.a, z.b, z.c, z.d};
      int idx = -1;
      for (int j = 0; j < 4; j++) if (cf[j]) idx = j;
      if (nz != 1 || (cf[idx] != 1 && cf[idx] != -1)) { d.unit = 0; d.ph[i] = -1; continue; }
      d.ph[i] = (int8_t)(idx + (cf[idx] < 0 ? 4 : 0));
    }
    // a Clifford gate's Pauli transfer matrix is a signed permutation, so a child's T bound (the smallest
    // sqrt2-valuation over the transfer matrix of the residual) is its parent's; a gate on one side of a cut
    // leaves that cut's operator-Schmidt rank unchanged.  Packed cut needs take 3 bits each in the node's
    // bound word, so at most BW_MAXCUTS cuts are carried.
    const int sde = gate_ptm_sde(h);
    d.tdel = sde >= 0 && sde < 255 ? sde : 255;
    for (const Zq &z : h.inv) terms += (z.a | z.b | z.c | z.d) != 0;
    columns += d.L;
    qubits += h.nq;
    d.cutloc = 0;
    d.cdel = 0;
    if ((int)s.cutmask.size() <= BW_MAXCUTS)
      for (size_t i = 0; i < s.cutmask.size(); i++) {
        if ((d.mask & s.cutmask[i]) == 0 || (d.mask & ~s.cutmask[i]) == 0) d.cutloc |= 1 << i;
        const int sr = gate_cut_rank(h, s.cutmask[i]);
        int del = 0;
        while (del < 7 && (1 << del) < sr) del++;
        d.cdel |= (sr < 1 ? 7 : del) << (3 * i);
      }
  }
  c->avg_terms = columns > 0 ? terms / columns : 1.0;
  c->avg_qubits = G > 0 ? qubits / G : 1.0;
  // T-bound classes: non-Clifford candidates whose children always have equal T bounds (same_t_bound), so a
  // parent's expansion computes the bound once per class
  {
    std::vector<int> cls(G, -1);
    int ncls = 0;
    for (int g = 0; g < G; g++) {
      if (dg[g].tdel == 0 || cls[g] >= 0) continue;
      std::vector<int> mem{g};
      for (int h2 = g + 1; h2 < G; h2++)
        if (dg[h2].tdel != 0 && cls[h2] < 0 && same_t_bound(s.gates[g], s.gates[h2])) mem.push_back(h2);
      if (mem.size() < 2 || ncls >= TC_MAX) continue;
      for (int m : mem) cls[m] = ncls;
      ncls++;
    }
    for (int g = 0; g < G; g++) dg[g].cls = cls[g] + 1;
  }
  std::vector<int4> goal(N * N);
  for (int i = 0; i < N * N; i++) goal[i] = make_int4((int)s.goal[i].a, (int)s.goal[i].b, (int)s.goal[i].c, (int)s.goal[i].d);
  std::vector<int> cx = s.cxtable.empty() ? std::vector<int>{0} : s.cxtable;
  // every table in one device block (256-byte aligned sections), one copy
  std::vector<uint8_t> blob;
  std::vector<std::pair<void **, size_t>> at;
  auto add = [&](void **dst, const void *src, size_t bytes) {
    const size_t off = (blob.size() + 255) & ~(size_t)255;
    blob.resize(off + std::max<size_t>(bytes, 1), 0);
    if (bytes) std::memcpy(blob.data() + off, src, bytes);
    at.push_back({dst, off});
  };
  add((void **)&c->d_gates, dg.data(), dg.size() * sizeof(DevGate));
  add((void **)&c->d_bad2, s.bad2.data(), s.bad2.size());
  add((void **)&c->d_bad3, s.bad3.data(), s.bad3.size() * 4);
  add((void **)&c->d_goal, goal.data(), goal.size() * sizeof(int4));
  add((void **)&c->d_cx, cx.data(), cx.size() * 4);
  add((void **)&c->d_symperm, c->grp.bperm.data(), c->grp.bperm.size());
  add((void **)&c->d_symconj, c->grp.conj.data(), c->grp.conj.size());
  // goal pre-images of every candidate, and the coefficient limit below which no child leaves int32: a child
  // coefficient is a sum over the gate column of parent coefficients times the column's Z[w] coefficients
  std::vector<int4> xg((size_t)G * N * N, make_int4(0, 0, 0, 0));
  std::vector<uint64_t> xgm(G, 0);
  std::vector<int> xgk(G, -1);
  uint64_t gmax = 1;
  std::vector<HostMat> pre;
  std::vector<char> have;
  c->goal_skip = goal_preimages(s, pre, have);
  for (int g = 0; g < G; g++) {
    const HostGate &h = s.gates[g];
    const HostMat &X = pre[g];
    if (have[g]) {
      xgk[g] = X.k;
      for (int i = 0; i < N * N; i++) {
        const Zq &z = X.e[i];
        xg[(size_t)g * N * N + i] = make_int4((int)z.a, (int)z.b, (int)z.c, (int)z.d);
        if (z.a | z.b | z.c | z.d) xgm[g] |= 1ull << i;
      }
    }
    const int L = 1 << h.nq;
    for (int lc = 0; lc < L; lc++) {
      uint64_t col = 0;
      for (int m = 0; m < L; m++) {
        const Zq &z = h.inv[m * L + lc];
        col += (uint64_t)(std::llabs(z.a) + std::llabs(z.b) + std::llabs(z.c) + std::llabs(z.d));
      }
      gmax = std::max(gmax, col);
    }
  }
  add((void **)&c->d_xg, xg.data(), xg.size() * sizeof(int4));
  add((void **)&c->d_xgm, xgm.data(), xgm.size() * 8);
  add((void **)&c->d_xgk, xgk.data(), xgk.size() * 4);
  c->spec_blob.need(blob.size());
  chz::copy_sync(c->spec_blob.p, blob.data(), blob.size(), hipMemcpyHostToDevice, c->stream);
  for (auto &d : at) *d.first = c->spec_blob.p + d.second;
  KSpec &k = c->ks;
  std::memset(&k, 0, sizeof k);
  k.n = s.n; k.G = G; k.depth = c->depth; k.standard = s.standard; k.lite = s.lite; k.tdiv = s.tdiv;
  k.gk = s.gk; k.nsym = c->grp.size(); k.ncuts = (int)s.cutmask.size(); k.have_table = !s.cxtable.empty();
  for (int i = 0; i < k.ncuts; i++) { k.cutmask[i] = s.cutmask[i]; k.cutsize[i] = s.cutsize[i]; k.rad[i] = s.rad[i]; }
  // the goal is the identity: exponent 0, T bound 0, rank-1 cuts, no support
  k.pre = (s.standard || s.lite) && s.gk == 0 && s.tdiv > 0;
  for (int i = 0; i < N * N; i++) {
    const Zq &z = s.goal[i];
    if (z.a != (i / N == i % N) || z.b || z.c || z.d) k.pre = 0;
  }
  if (k.have_table && s.cxtable[0] != 0) k.pre = 0;     // the goal needs no cut, but its cut bound is not 0
  // a cut bound from lowered needs is a lower bound only if the table never decreases when a need grows
  k.cx_mono = 1;
  k.ncx = (int)s.cxtable.size();
  k.cut1 = k.ncuts <= std::min(CSRC_MAX, BW_MAXCUTS);
  for (int i = 0; i < k.ncuts; i++) k.cut1 = k.cut1 && k.cutsize[i] == 1 && k.rad[i] == 3 && k.n > 1;
  k.cxlds = s.cxtable.size() <= (size_t)CXL_MAX;
  for (int v : s.cxtable) if (v < 0 || v > 255) k.cxlds = 0;
  if (k.have_table) {
    size_t total = 1;
    for (int i = 0; i < k.ncuts; i++) total *= (size_t)s.rad[i];
    if (total != s.cxtable.size()) k.cx_mono = 0;
    for (size_t idx = 0; k.cx_mono && idx < total; idx++) {
      size_t rest = idx, mult = 1;
      for (int i = 0; i < k.ncuts; i++) {
        const size_t nd = rest % (size_t)s.rad[i];
        rest /= (size_t)s.rad[i];
        if (nd + 1 < (size_t)s.rad[i] && s.cxtable[idx + mult] < s.cxtable[idx]) k.cx_mono = 0;
        mult *= (size_t)s.rad[i];
      }
    }
  }
  k.gates = c->d_gates; k.bad2 = c->d_bad2; k.bad3 = c->d_bad3; k.goal = c->d_goal; k.cxtable = c->d_cx;
  k.goalnz = 0;
  for (int i = 0; i < N * N; i++) {
    const Zq &z = s.goal[i];
    if (z.a || z.b || z.c || z.d) k.goalnz |= 1ull << i;
  }
  k.symperm = c->d_symperm; k.symconj = c->d_symconj;
  k.xg = c->d_xg; k.xgm = c->d_xgm; k.xgk = c->d_xgk;
  k.maglim = (uint32_t)(0x7fffffffull / gmax);
  k.cjm = 0;
  for (int y = 0; y < k.nsym && y < 16; y++) k.cjm |= (uint32_t)(c->grp.conj[y] != 0) << y;
  std::vector<SpecTabs> tabs(1);
  build_level_tabs(tabs[0], dg, k, c->grp, s);
  c->max_ik = 0;
  bool two_terms = true;
  for (int g = 0; g < G; g++) {
    c->max_ik = std::max(c->max_ik, dg[g].ik);
    two_terms = two_terms && (tabs[0].level.head[g].w & 1u);
  }
  c->std_spec = s.standard && !s.lite && k.pre && k.cut1 && k.ncuts == (k.n == 3 ? 3 : 1) && k.n > 1 && k.have_table &&
                k.cxlds && k.cx_mono && two_terms;
  c->tcols = c->std_spec && k.n == 3;
  c->ktab.need(sizeof(SpecTabs));
  chz::copy_sync(c->ktab.p, tabs.data(), sizeof(SpecTabs), hipMemcpyHostToDevice, c->stream);
  k.ktab = (const uint4 *)c->ktab.p;
}

// The candidates' column maps (gate_columns), formed when a frontier first carries T columns: until then no kernel reads
// them, and forming them took a seventh of a one-gate search on a context of its own (0.49 ms, 0.42 without)
static void form_columns(chz_ctx *c) {
  if (c->cols_formed) return;
  std::vector<uint8_t> col_src((size_t)MAXG * 64, 255);
  std::vector<uint64_t> keep_cols(MAXG, 0);
  for (int g = 0; g < c->hs.G(); g++) {
    std::vector<int> src;
    gate_columns(c->hs.gates[g], 3, src);
    for (int b = 0; b < 64; b++)
      if (src[b] >= 0) {
        col_src[g * 64 + b] = (uint8_t)src[b];
        keep_cols[g] |= 1ull << src[b];
      }
  }
  copy_sync(c->ktab.p + offsetof(SpecTabs, col_src), col_src.data(), col_src.size(), hipMemcpyHostToDevice, c->stream);
  copy_sync(c->ktab.p + offsetof(SpecTabs, level) + offsetof(LevelTabs, keep_cols), keep_cols.data(), keep_cols.size() * 8,
            hipMemcpyHostToDevice, c->stream);
  c->cols_formed = true;
}

// a new search of the batch: the depth-0 cases end at once (src/cheese.cu:1794-1801), the rest wait to join
// the frontier as roots at the next step
static int batch_add_parsed(chz_ctx *c, const HostSpec &hs, int depth, int tag) {
  const int N = hs.N(), E = N * N;
  chz_event ev{};
  ev.tag = tag;
  ev.kind = 1;
  for (int i = 0; i < E; i++) {
    const Zq &z = hs.target[i];
    if (z.a != (int32_t)z.a || z.b != (int32_t)z.b || z.c != (int32_t)z.c || z.d != (int32_t)z.d) {
      set_err("target coefficients exceed int32");
      ev.result.rc = 4;
      c->events.push_back(ev);
      return 0;
    }
  }
  HostMat U;
  U.e = hs.target;
  U.k = hs.tk;
  if (!c->nogoal && host_equal(U, c->hs.goal, c->hs.gk)) { ev.result.rc = 0; c->events.push_back(ev); return 0; }
  if (depth <= 0) { ev.result.rc = 1; c->events.push_back(ev); return 0; }
  // a free instance slot: not held by a live search
  std::vector<bool> used(c->nslots + c->binst.size() + 1, false);
  for (const BInst &b : c->binst)
    if (b.live) {
      used[b.slot] = true;
      c->shared_steps = true;      // the batch now steps more than one search
    }
  int slot = 0;
  while (used[slot]) slot++;
  try {
    HIPCHK(hipSetDevice(c->device));
    reserve_slots(c, slot + 1);
  } catch (DeviceError &) {
    return 5;
  }
  int bi = -1;
  for (size_t i = 0; i < c->binst.size(); i++) if (!c->binst[i].live) { bi = (int)i; break; }
  if (bi < 0) { c->binst.emplace_back(); bi = (int)c->binst.size() - 1; }
  BInst &b = c->binst[bi];
  b = BInst{};
  b.tag = tag;
  b.depth = depth;
  b.slot = slot;
  b.live = true;
  b.t0 = now_s();
  Pending q;
  q.inst = bi;
  q.k = b.k = hs.tk;
  b.reducible = hs.tk > 0;
  for (const Zq &z : hs.target) {
    for (long long v : {(long long)z.a, (long long)z.b, (long long)z.c, (long long)z.d}) b.coef = std::max(b.coef, (uint32_t)std::llabs(v));
    b.reducible = b.reducible && !((z.a - z.c) & 1) && !((z.b - z.d) & 1);
  }
  q.U.resize(E);
  for (int i = 0; i < E; i++) {
    const Zq &z = hs.target[i];
    q.U[i] = make_int4((int)z.a, (int)z.b, (int)z.c, (int)z.d);
  }
  c->pending.push_back(std::move(q));
  return 0;
}

#include "table_join.h"

}  // namespace chz

// ------------------------------------------------------------------------------------------------------
// C ABI

extern "C" {

const char *chz_last_error(void) { return chz::get_err(); }

int chz_open(const char *spec_text, size_t len, const chz_opts *opts, chz_ctx **out) {
  *out = nullptr;
  std::unique_ptr<chz_ctx> c(new chz_ctx());
  std::string err;
  if (const int prc = chz::parse_spec(std::string(spec_text, len), c->hs, err)) { chz::set_err(err); return prc; }
  chz_opts o{-1, 1, 1, 0, 0, 0};
  if (opts) o = *opts;
  c->opts = o;
  c->depth = o.depth >= 0 ? o.depth : c->hs.depth;
  c->ev.mask = o.profile ? ~0u : 0u;
  if (c->depth > CHZ_DMAX) { chz::set_err("depth > 48"); return 3; }
  if (c->hs.states) { chz::set_err("state targets are not supported by this build"); return 3; }
  if (c->hs.n < 1 || c->hs.n > 3) { chz::set_err("n = " + std::to_string(c->hs.n) + " not built (1..3)"); return 3; }
  if (c->hs.truncated) { chz::set_err("malformed spec"); return 2; }
  if ((int)c->hs.target.size() != c->hs.N() * c->hs.N()) { chz::set_err("spec has no target"); return 2; }
  // symmetry classes: not with --mitm, whose join compares exact residuals (src/cheese.cu:1786)
  c->grp = chz::build_symmetry(c->hs, o.sym != 0 && !o.mitm);
  if (o.table < 0 || o.table > CHZ_DMAX) { chz::set_err("--table K outside 0..48"); return 3; }
  // default occupancy: groups of less than a wave spill above 4 waves per SIMD
  if (c->hs.n < 3)
    for (auto &sc : c->sched) sc.var = 0;
  else
    // n = 3 defaults per level-size bucket (log2 of the parents in a launch), from the autotuner's winners on the
    // Toffoli proofs of budgets 9 to 14 on MI355X.  The expansion is bound by instruction issue, with waits on LDS and on
    // the parents' loads between: from 4K parents on 6 waves per SIMD (80 registers) win, budget-13 levels of a million
    // parents take 4.7 ms instead of 5.4 with 5.  Below, the waves have a parent or less each, and it is the longest
    // chain that counts: a parent's candidates are split over lane groups, up to 512 parents down to one or two
    // candidates each at the variant with the most registers
    for (int b = 0; b < (int)(sizeof c->sched / sizeof c->sched[0]); b++) {
      chz_ctx::Sched &sc = c->sched[b];
      if (b <= 8) { sc.var = 0; sc.tw = 16384; }
      else if (b <= 11) { sc.var = 1; sc.tw = 8192; }
      else if (b <= 14) { sc.var = 2; sc.cap = 4096; sc.tw = b == 12 ? 8192 : 16384; }
      else { sc.var = 2; sc.cap = b == 15 ? 8192 : 16384; }
    }
  try {
    c->device = o.device;
    HIPCHK(hipSetDevice(o.device));
    HIPCHK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
    chz::StreamScope scope(c->stream, &c->retired);
    chz::upload_spec(c.get());
  } catch (chz::DeviceError &) {
    return 5;
  }
  *out = c.release();
  return 0;
}

int chz_run(chz_ctx *c, chz_level_cb cb, void *user, chz_result *out) {
  chz_result tmp{};
  chz_result *res = out ? out : &tmp;
  std::memset(res, 0, sizeof *res);
  if (chz_batch_live(c)) { chz::set_err("the context's batch holds searches"); return res->rc = 3; }
  for (int f = 0; f < chz::K_NFAM; f++) { c->k_launch[f] = 0; c->k_ms[f] = 0; c->k_work[f] = 0; }
  for (double &v : c->k_stage) v = 0;
  c->events.clear();
  res->split_kind = 0;
  res->split[0] = res->split[1] = -1;
  if (c->opts.mitm || c->opts.table > 0) {   // --mitm takes precedence, as in the reference (src/cheese.cu:1803)
    try {
      HIPCHK(hipSetDevice(c->device));
      chz::StreamScope scope(c->stream, &c->retired);
      switch (c->hs.n) {
        case 1: return c->opts.mitm ? chz::run_mitm<1>(c, cb, user, res) : chz::run_table<1>(c, cb, user, res);
        case 2: return c->opts.mitm ? chz::run_mitm<2>(c, cb, user, res) : chz::run_table<2>(c, cb, user, res);
        default: return c->opts.mitm ? chz::run_mitm<3>(c, cb, user, res) : chz::run_table<3>(c, cb, user, res);
      }
    } catch (chz::DeviceError &) {
      return res->rc = 5;
    }
  }
  const int rc0 = chz::batch_add_parsed(c, c->hs, c->depth, 0);
  if (rc0) return res->rc = rc0;
  while (true) {
    chz_event e;
    bool done = false;
    while (!c->events.empty()) {
      e = c->events.front();
      c->events.pop_front();
      if (e.kind == 0) { if (cb) cb(&e.level, user); }
      else { *res = e.result; done = true; }
    }
    if (done) return res->rc;
    if (const int rc = chz_batch_step(c)) return res->rc = rc;
  }
}

// the expansion schedule per level-size bucket, chosen by timing every candidate schedule on this context's own
// search (reps runs each); the fastest mean launch time per bucket wins.  Per-level results do not depend on
// the schedule.  out (may be NULL) receives the chosen table as JSON text.
int chz_tune(chz_ctx *c, int reps, char *out, size_t cap) {
  if (chz_batch_live(c)) { chz::set_err("the context's batch holds searches"); return 3; }
  const int vars[3] = {0, 1, 2}, caps[3] = {4096, 8192, 16384}, tws[5] = {2048, 4096, 8192, 16384, 32768};
  std::vector<chz_ctx::Sched> cands;
  for (int v : vars) for (int cp : caps) for (int tw : tws) { chz_ctx::Sched s; s.var = v; s.cap = cp; s.tw = tw; cands.push_back(s); }
  std::vector<std::vector<double>> sum(cands.size(), std::vector<double>(32, 0.0));
  std::vector<std::vector<int>> num(cands.size(), std::vector<int>(32, 0));
  try {
    HIPCHK(hipSetDevice(c->device));
    for (size_t k = 0; k < cands.size(); k++) {
      c->tuning = true;
      c->force = cands[k];
      for (int r = 0; r < std::max(1, reps); r++) {
        chz_result res{};
        const int rc = chz_run(c, nullptr, nullptr, &res);
        if (rc >= 2) { c->tuning = false; return rc; }
        HIPCHK(hipStreamSynchronize(c->stream));
        for (auto &te : c->tune_ev) {
          float ms = 0;
          HIPCHK(hipEventElapsedTime(&ms, te.second.first, te.second.second));
          sum[k][te.first] += ms;
          num[k][te.first]++;
          c->ev.pool.push_back(te.second.first);
          c->ev.pool.push_back(te.second.second);
        }
        c->tune_ev.clear();
      }
    }
  } catch (chz::DeviceError &) {
    c->tuning = false;
    return 5;
  }
  c->tuning = false;
  std::string js = "{";
  bool first = true;
  for (int b = 0; b < 32; b++) {
    int best = -1;
    for (size_t k = 0; k < cands.size(); k++)
      if (num[k][b] && (best < 0 || sum[k][b] / num[k][b] < sum[best][b] / num[best][b])) best = (int)k;
    if (best < 0) continue;
    c->sched[b] = cands[best];
    char buf[128];
    std::snprintf(buf, sizeof buf, "%s\"%d\": {\"waves_per_eu\": %d, \"grid_cap\": %d, \"split_waves\": %d, \"ms\": %.4f}",
                  first ? "" : ", ", b, cands[best].var + 4, cands[best].cap, cands[best].tw, sum[best][b] / num[best][b]);
    js += buf;
    first = false;
  }
  js += "}";
  if (out && cap) { std::strncpy(out, js.c_str(), cap - 1); out[cap - 1] = 0; }
  return 0;
}

int chz_batch_add(chz_ctx *c, const char *spec_text, size_t len, int depth, int tag) {
  chz::HostSpec hs;
  std::string err;
  if (const int prc = chz::parse_spec(std::string(spec_text, len), hs, err)) { chz::set_err(err); return prc; }
  if (hs.truncated) { chz::set_err("malformed spec"); return 2; }
  if (hs.states) { chz::set_err("state targets are not supported by this build"); return 3; }
  if ((int)hs.target.size() != hs.N() * hs.N()) { chz::set_err("spec has no target"); return 2; }
  if (!chz::same_gate_set(hs, c->hs)) { chz::set_err("the spec's gate set differs from the batch's"); return 3; }
  const int d = depth >= 0 ? depth : hs.depth;
  if (d > CHZ_DMAX) { chz::set_err("depth > 48"); return 3; }
  return chz::batch_add_parsed(c, hs, d, tag);
}

int chz_batch_step(chz_ctx *c) {
  try {
    HIPCHK(hipSetDevice(c->device));
    chz::StreamScope scope(c->stream, &c->retired);
    switch (c->hs.n) {
      case 1: chz::batch_step<1>(c); break;
      case 2: chz::batch_step<2>(c); break;
      case 3: chz::batch_step<3>(c); break;
    }
    return 0;
  } catch (chz::DeviceError &) {
    return 5;
  }
}

void chz_batch_set_budget(chz_ctx *c, double bytes) { c->mem_budget = bytes > 0 ? bytes : 0; }

long long chz_batch_waits(const chz_ctx *c) { return c->carried_levels; }

long long chz_batch_frontier(chz_ctx *c, long long max, long long stride, int *paths, int *lens, uint32_t *bw,
                             int *tags) {
  if (stride < 1) stride = 1;
  long long n = 0;
  try {
    HIPCHK(hipSetDevice(c->device));
    chz::StreamScope scope(c->stream, &c->retired);
    HIPCHK(hipStreamSynchronize(c->stream));
    std::vector<int> seq;
    for (long long j = 0; j < c->m && n < max; j += stride, n++) {
      uint32_t w = 0, slot = 0;
      chz::copy_sync(&w, c->pb[c->cur].p + j, 4, hipMemcpyDeviceToHost, c->stream);
      chz::copy_sync(&slot, c->finst[c->cur].p + j, 4, hipMemcpyDeviceToHost, c->stream);
      // the node's gates from its root: the tree walked up from the current level, as walk_circuits does
      seq.clear();
      uint32_t i = (uint32_t)j;
      for (int s = c->gstep; s >= 0 && c->tree_par[s]; s--) {
        uint32_t par;
        uint8_t g;
        chz::copy_sync(&par, c->tree_par[s] + i, 4, hipMemcpyDeviceToHost, c->stream);
        if (par == chz::NO_PARENT) break;
        chz::copy_sync(&g, c->tree_gate[s] + i, 1, hipMemcpyDeviceToHost, c->stream);
        if (g != chz::CARRY_GATE) seq.push_back(g);
        i = par;
      }
      std::reverse(seq.begin(), seq.end());
      const int len = (int)std::min<size_t>(seq.size(), CHZ_DMAX);
      for (int t = 0; t < len; t++) paths[(size_t)n * CHZ_DMAX + t] = seq[t];
      lens[n] = len;
      bw[n] = w;
      tags[n] = -1;
      for (const chz::BInst &b : c->binst)
        if (b.live && (uint32_t)b.slot == slot) tags[n] = b.tag;
    }
  } catch (chz::DeviceError &) {
    return -1;
  }
  return n;
}

int chz_batch_events(chz_ctx *c, chz_event *out, int max) {
  int k = 0;
  while (k < max && !c->events.empty()) { out[k++] = c->events.front(); c->events.pop_front(); }
  return k;
}

int chz_batch_live(const chz_ctx *c) {
  int n = 0;
  for (const chz::BInst &b : c->binst) n += b.live;
  return n;
}

long long chz_batch_nodes(const chz_ctx *c) {
  long long n = c->m;
  return n + (long long)c->pending.size();
}

int chz_num_gates(const chz_ctx *c) { return c->hs.G(); }
int chz_num_qubits(const chz_ctx *c) { return c->hs.n; }
int chz_depth(const chz_ctx *c) { return c->depth; }
int chz_sym_size(const chz_ctx *c) { return c->grp.size(); }
const char *chz_gate_name(const chz_ctx *c, int g) {
  return g >= 0 && g < c->hs.G() ? c->hs.gates[g].name.c_str() : "";
}

int chz_profile(const chz_ctx *c, const char **names, double *seconds, int n) {
  int j = 0;
  for (int f = 0; f < chz::K_NFAM && j < n; f++, j++) {
    if (names) names[j] = chz::k_names[f];
    if (seconds) seconds[j] = c->k_ms[f] / 1000.0;
  }
  return j;
}

unsigned chz_time_kernels(chz_ctx *c, unsigned families) {
  const unsigned prev = c->ev.mask;
  c->ev.mask = families;
  return prev;
}

int chz_expand_stages(const chz_ctx *c, double *out) {
  for (int i = 0; i < 6; i++) out[i] = c->k_stage[i];
  return 6;
}

int chz_kernel_stats(const chz_ctx *c, chz_kstat *out, int n) {
  int j = 0;
  for (int f = 0; f < chz::K_NFAM && j < n; f++, j++) {
    out[j].name = chz::k_names[f];
    out[j].launches = c->k_launch[f];
    out[j].ms = c->k_ms[f];
    out[j].work = c->k_work[f];
  }
  return j;
}

static int verify_hs(const chz::HostSpec &hs, const int *circuit, int len) {
  // product of the forward gate matrices, gate 1 first, compared exactly with the target (verify.py:20-33)
  const int n = hs.n, N = 1 << n;
  chz::HostMat P;
  P.e.assign(N * N, chz::Zq{0, 0, 0, 0});
  for (int i = 0; i < N; i++) P.e[i * N + i] = chz::Zq{1, 0, 0, 0};
  for (int j = 0; j < len; j++) {
    if (circuit[j] < 0 || circuit[j] >= hs.G()) return -1;
    // P <- g P via (P^dag g^dag)^dag: apply g on the left with its forward matrix
    const chz::HostGate &g = hs.gates[circuit[j]];
    const int L = 1 << g.nq;
    int mask = 0;
    for (int q = 0; q < g.nq; q++) mask |= 1 << g.q[q];
    std::vector<chz::Zq> out(N * N, chz::Zq{0, 0, 0, 0});
    for (int r = 0; r < N; r++) {
      int lr = 0;
      for (int q = 0; q < g.nq; q++) lr |= ((r >> g.q[q]) & 1) << q;
      const int base = r & ~mask;
      for (int m = 0; m < L; m++) {
        const chz::Zq gm = g.fwd[lr * L + m];
        if (!(gm.a | gm.b | gm.c | gm.d)) continue;
        int x = base;
        for (int q = 0; q < g.nq; q++) if ((m >> q) & 1) x |= 1 << g.q[q];
        for (int col = 0; col < N; col++) {
          const chz::Zq v = P.e[x * N + col];
          chz::Zq &o = out[r * N + col];
          o.a += gm.a * v.a - gm.b * v.d - gm.c * v.c - gm.d * v.b;
          o.b += gm.a * v.b + gm.b * v.a - gm.c * v.d - gm.d * v.c;
          o.c += gm.a * v.c + gm.b * v.b + gm.c * v.a - gm.d * v.d;
          o.d += gm.a * v.d + gm.b * v.c + gm.c * v.b + gm.d * v.a;
        }
      }
    }
    P.e.swap(out);
    P.k += g.gk;
    while (P.k > 0) {
      bool all = true;
      for (auto &z : P.e) if (((z.a - z.c) & 1) || ((z.b - z.d) & 1)) { all = false; break; }
      if (!all) break;
      for (auto &z : P.e) z = chz::Zq{(z.b - z.d) / 2, (z.a + z.c) / 2, (z.b + z.d) / 2, (z.c - z.a) / 2};
      P.k--;
    }
  }
  return chz::host_equal(P, hs.target, hs.tk) ? 1 : 0;
}

int chz_verify(const chz_ctx *c, const int *circuit, int len) { return verify_hs(c->hs, circuit, len); }

int chz_verify_spec(const char *spec_text, size_t len, const int *circuit, int n) {
  chz::HostSpec hs;
  std::string err;
  if (chz::parse_spec(std::string(spec_text, len), hs, err) || hs.truncated ||
      (int)hs.target.size() != hs.N() * hs.N()) {
    chz::set_err(err.empty() ? "malformed spec" : err);
    return -2;
  }
  return verify_hs(hs, circuit, n);
}

void chz_close(chz_ctx *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  chz::free_tree(c);
  for (int b = 0; b < 2; b++) {
    c->res[b].release(); c->pk[b].release(); c->g1[b].release(); c->g2[b].release();
    c->pb[b].release(); c->tm[b].release();
    c->sk[b].release(); c->sv[b].release();
  }
  c->finst[0].release(); c->finst[1].release(); c->ctl.release(); c->gflag.release();
  c->scan_tmp.release();
  chz::settle(c->retired);
  c->pin.release();
  c->pin_io.release();
  for (auto &g : c->sgraph) if (g.exec) { (void)hipGraphExecDestroy(g.exec); g.exec = nullptr; }
  c->status.release(); c->kept.release(); c->keys.release(); c->surv_o.release(); c->surv_key.release();
  c->surv_bw.release();
  c->info.release(); c->bcount.release(); c->hist.release(); c->kidx.release();
  c->spec_blob.release();
  c->ktab.release();
  if (c->gt) { c->gt->release(); delete c->gt; c->gt = nullptr; }
  c->gt_keys.release(); c->gt_hit.release(); c->gt_cost.release(); c->gt_best.release();
  c->ev.destroy();
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

}  // extern "C"
