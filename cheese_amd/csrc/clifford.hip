// The n-qubit Clifford group (n <= 3) tabulated on one MI355X: breadth-first search by gate count from the
// identity into an open-addressing HBM hash table (tableau -> minimal gate count), batched distance queries
// and optimal-word read-back.  Reference behaviour: src/clifford.cu:41-166 (tableaux, table, BFS),
// :207-210 (batched find), :251-283 (BFS driver, group-order check), :344-372 (read-back).
//
// Table layout.  A tableau is a symplectic matrix and a sign per row; a gate changes the matrix independently of the
// signs and XORs the signs with a vector that depends on the matrix alone.  So the group is (symplectic matrices) x (sign
// vectors): 1,451,520 x 64 at 3 qubits.  The matrices are numbered (in the order of their tableaux, by unranking), a
// hash table of 2^22 8-byte slots maps a matrix to its number, and the distances of its 64 sign vectors are four 64-bit
// planes, bit s of plane k being bit k of the distance of sign vector s (distances are at most 13).  78 MB instead of
// 1.07 GB for a hash table of whole tableaux, which the 256 MB last-level cache holds.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cstring>
#include <mutex>
#include <sstream>
#include <string>
#include <vector>

#include "../../include/cheese_hip.h"
#include "host.h"
#include "primitives.h"

// Device allocations of the Clifford table go through the process-wide capture lock: another thread (the request
// server's gate-count engines) may be capturing a level step, and hipFree synchronises the device.
static hipError_t cl_malloc(void **p, size_t bytes) {
  std::lock_guard<std::recursive_mutex> g(chz::capture_mu());
  return hipMalloc(p, bytes);
}
static hipError_t cl_free(void *p) {
  std::lock_guard<std::recursive_mutex> g(chz::capture_mu());
  return hipFree(p);
}

namespace chz_cl {

struct Gates { int n, ng; int k[32], a[32], b[32]; };   // gate set: H, S, Sdg, X, Z per qubit, then CX pairs

static Gates gate_set(int n) {
  Gates G{};
  G.n = n;
  for (int q = 0; q < n; q++)
    for (int k = 0; k < 5; k++) { G.k[G.ng] = k; G.a[G.ng] = q; G.b[G.ng] = 0; G.ng++; }
  for (int a = 0; a < n; a++)
    for (int b = 0; b < n; b++)
      if (a != b) { G.k[G.ng] = 5; G.a[G.ng] = a; G.b[G.ng] = b; G.ng++; }
  return G;
}

// Tableau: 2n rows (images of X_0..X_{n-1}, Z_0..Z_{n-1}), row = x | z << n | sign << 2n, for the Hermitian
// Pauli (-1)^sign i^(x.z) X^x Z^z.  Gate kinds: 0 H, 1 S, 2 Sdg, 3 X, 4 Z, 5 CX a->b, 6 Y.
__host__ __device__ inline uint32_t conj_row(uint32_t w, int n, int k, int a, int b) {
  const uint32_t nm = (1u << n) - 1;
  uint32_t x = w & nm, z = (w >> n) & nm, r = (w >> (2 * n)) & 1;
  const uint32_t xa = (x >> a) & 1, za = (z >> a) & 1;
  if (k == 0) { r ^= xa & za; x = (x & ~(1u << a)) | (za << a); z = (z & ~(1u << a)) | (xa << a); }
  else if (k == 1) { r ^= xa & za; z ^= xa << a; }
  else if (k == 2) { r ^= xa & (za ^ 1); z ^= xa << a; }
  else if (k == 3) { r ^= za; }
  else if (k == 4) { r ^= xa; }
  else if (k == 5) {
    const uint32_t xb = (x >> b) & 1, zb = (z >> b) & 1;
    r ^= xa & zb & (xb ^ za ^ 1);
    x ^= xa << b;
    z ^= zb << a;
  } else { r ^= xa ^ za; }
  return x | (z << n) | (r << (2 * n));
}
__host__ __device__ inline uint64_t apply(uint64_t T, int n, int k, int a, int b) {   // gate after the Clifford T
  const int rb = 2 * n + 1;
  const uint64_t rm = (1ull << rb) - 1;
  uint64_t out = 0;
  for (int i = 0; i < 2 * n; i++) out |= (uint64_t)conj_row((uint32_t)((T >> (i * rb)) & rm), n, k, a, b) << (i * rb);
  return out;
}
__host__ __device__ inline uint64_t identity(int n) {
  const int rb = 2 * n + 1;
  uint64_t T = 0;
  for (int i = 0; i < n; i++) { T |= (uint64_t)(1u << i) << (i * rb); T |= (uint64_t)(1u << (n + i)) << ((n + i) * rb); }
  return T;
}
__host__ __device__ inline int inv_kind(int k) { return k == 1 ? 2 : k == 2 ? 1 : k; }

__host__ __device__ inline uint64_t hmix(uint64_t x) {
  x ^= x >> 31; x *= 0x7fb5d329728ea185ull;
  x ^= x >> 27; x *= 0x81dadef4bc2dd44dull;
  return x ^ (x >> 33);
}

// bits 2n of every row: the signs
__host__ __device__ inline uint64_t sign_mask(int n) {
  uint64_t m = 0;
  for (int i = 0; i < 2 * n; i++) m |= 1ull << (i * (2 * n + 1) + 2 * n);
  return m;
}
// the rows' signs, row i in bit i
__host__ __device__ inline uint32_t signs_of(uint64_t T, int n) {
  uint32_t s = 0;
  for (int i = 0; i < 2 * n; i++) s |= (uint32_t)((T >> (i * (2 * n + 1) + 2 * n)) & 1) << i;
  return s;
}

constexpr int IDX_BITS = 21;       // matrix numbers; tableaux have at most 42 bits

struct Table {
  unsigned long long *slot;        // tableau without signs << 21 | number; 0 = empty (no tableau is 0)
  uint32_t smask;                  // slots - 1
  const ulonglong2 *planes;        // two per matrix: planes 0, 1 and 2, 3
  const uint8_t *dmin;             // per matrix, the smallest distance of its sign vectors
  int n;
};

// number of the symplectic matrix with this sign-free tableau, -1 when it is none
__device__ inline int find_sym(const Table &T, uint64_t key) {
  for (uint32_t b = (uint32_t)hmix(key) & T.smask;; b = (b + 1) & T.smask) {
    const unsigned long long v = T.slot[b];
    if (!v) return -1;
    if (v >> IDX_BITS == key) return (int)(v & ((1u << IDX_BITS) - 1));
  }
}
__device__ inline int plane_dist(ulonglong2 p, ulonglong2 q, uint32_t s) {
  return (int)(((p.x >> s) & 1) | ((p.y >> s) & 1) << 1 | ((q.x >> s) & 1) << 2 | ((q.y >> s) & 1) << 3);
}
// distance of a tableau, -1 when it is none
__device__ inline int find1(const Table &T, uint64_t key) {
  const int i = find_sym(T, key & ~sign_mask(T.n));
  return i < 0 ? -1 : plane_dist(T.planes[2 * i], T.planes[2 * i + 1], signs_of(key, T.n));
}

// ---- numbering.  A tableau's rows are chosen from the last to the first (the most significant first): row 2n - 1 any
// nonzero vector, each further Z image a vector that commutes with those before it and is independent of them, each X
// image a vector that anticommutes with its Z image and commutes with the other rows.  However the rows before it were
// chosen, a row has the same number of choices (63, 30, 12, 8, 4, 2 at 3 qubits), so a mixed-radix number with a row's
// choice, in increasing order of its vector, as digit lists the matrices in the order of their tableaux.  With the
// row's sign above its choice in every digit the number lists all tableaux in order.
template <int NQ> struct Num {
  static constexpr int M = 2 * NQ;
  static constexpr uint64_t FULL = M == 6 ? ~0ull : (1ull << (1 << M)) - 1;     // all vectors
  // choices of the k-th row chosen (row M - 1 - k)
  __host__ __device__ static constexpr uint32_t choices(int k) { return k < NQ ? (1u << (M - k)) - (1u << k) : 1u << (M - k); }
  __host__ __device__ static constexpr long long matrices() {
    long long t = 1;
    for (int k = 0; k < M; k++) t *= choices(k);
    return t;
  }
  static constexpr long long ORDER = matrices() << M;
  // vectors (as bits of a mask) that anticommute with v
  __host__ __device__ static uint64_t anti(uint32_t v) {
    constexpr uint64_t B[6] = {0xaaaaaaaaaaaaaaaaull, 0xccccccccccccccccull, 0xf0f0f0f0f0f0f0f0ull,
                               0xff00ff00ff00ff00ull, 0xffff0000ffff0000ull, 0xffffffff00000000ull};
    uint64_t m = 0;
#pragma unroll
    for (int i = 0; i < M; i++)
      if ((v >> ((i + NQ) % M)) & 1) m ^= B[i];
    return m & FULL;
  }
  // the mask with bit v ^ d in place of bit v
  __host__ __device__ static uint64_t shift(uint64_t m, uint32_t d) {
    constexpr uint64_t L[6] = {0x5555555555555555ull, 0x3333333333333333ull, 0x0f0f0f0f0f0f0f0full,
                               0x00ff00ff00ff00ffull, 0x0000ffff0000ffffull, 0x00000000ffffffffull};
#pragma unroll
    for (int i = 0; i < M; i++)
      if ((d >> i) & 1) m = ((m >> (1 << i)) & L[i]) | ((m & L[i]) << (1 << i));
    return m;
  }
  // place of the bit of m that r others lie below (halving; one by one, samples of the 3-qubit group took 38 us a call)
  __host__ __device__ static uint32_t nth_bit(uint64_t m, uint32_t r) {
    uint32_t at = 0;
#pragma unroll
    for (int w = 1 << (M - 1); w; w >>= 1) {
      const uint32_t c = (uint32_t)__builtin_popcountll(m >> at & ((1ull << w) - 1));
      const bool up = r >= c;
      r -= up ? c : 0u;
      at += up ? (uint32_t)w : 0u;
    }
    return at;
  }
  // the tableau whose k-th chosen row is choice r[k], row i signed by bit i of s
  __host__ __device__ static uint64_t tableau(const uint32_t (&r)[M], uint32_t s) {
    uint64_t an[M], span = 1, T = 0;
#pragma unroll
    for (int k = 0; k < M; k++) {
      const int row = M - 1 - k;
      uint64_t m = FULL;
#pragma unroll
      for (int j = 0; j < k; j++) m &= (M - 1 - j) == row + NQ ? an[j] : ~an[j];
      if (k < NQ) m &= ~span;
      const uint32_t v = nth_bit(m, r[k]);
      an[k] = anti(v);
      if (k < NQ) span |= shift(span, v);
      T |= (uint64_t)(v | ((s >> row) & 1) << M) << (row * (M + 1));
    }
    return T;
  }
  // matrices and tableaux that share their Z images (the rows chosen first): numbers differ below these
  __host__ __device__ static constexpr uint32_t x_matrices() {
    uint32_t t = 1;
    for (int k = NQ; k < M; k++) t *= choices(k);
    return t;
  }
  static constexpr uint32_t X_SYM = x_matrices(), X_ALL = X_SYM << NQ;
  static constexpr uint32_t Z_SYM = (uint32_t)(matrices() / X_SYM), Z_ALL = Z_SYM << NQ;
  // the number, among all tableaux, of the i-th matrix with signs s
  __host__ __device__ static uint64_t signed_number(uint32_t i, uint32_t s) {
    uint64_t e = 0, scale = 1;
#pragma unroll
    for (int k = M - 1; k >= 0; k--) {
      const uint32_t c = choices(k);
      e += scale * (i % c + ((s >> (M - 1 - k)) & 1) * c);
      scale *= 2 * c;
      i /= c;
    }
    return e;
  }
  // the i-th matrix's tableau, without signs
  __host__ __device__ static uint64_t matrix(uint32_t i) {
    uint32_t r[M];
#pragma unroll
    for (int k = M - 1; k >= 0; k--) { r[k] = i % choices(k); i /= choices(k); }
    return tableau(r, 0);
  }
  // the i-th tableau
  __host__ __device__ static uint64_t element(uint64_t i) {
    uint32_t r[M], s = 0;
#pragma unroll
    for (int k = M - 1; k >= 0; k--) {
      const uint32_t d = (uint32_t)(i % (2 * choices(k)));
      i /= 2 * choices(k);
      r[k] = d % choices(k);
      s |= (d / choices(k)) << (M - 1 - k);
    }
    return tableau(r, s);
  }
};

// ---- building the table.  Gates that change the matrix: H, S (Sdg with it) on each qubit, CX on each ordered pair.
__host__ __device__ constexpr int sym_gates(int n) { return 2 * n + n * (n - 1); }

template <int NQ> __global__ __launch_bounds__(256) void k_matrices(uint64_t *key, unsigned long long *slot, uint32_t smask) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint32_t)Num<NQ>::matrices()) return;
  const uint64_t T = Num<NQ>::matrix(i);
  key[i] = T;
  const unsigned long long v = (unsigned long long)T << IDX_BITS | i;
  for (uint32_t b = (uint32_t)hmix(T) & smask;; b = (b + 1) & smask)
    if (atomicCAS(&slot[b], 0ull, v) == 0ull) break;
}

// nb[g * count + i]: the matrix that matrix-changing gate g takes matrix i to (and from: each is its own inverse on the
// matrices)
template <int NQ> __global__ __launch_bounds__(256) void k_neighbours(Table T, const uint64_t *key, uint32_t *nb) {
  constexpr uint32_t C = (uint32_t)Num<NQ>::matrices();
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= C) return;
  const uint64_t t = key[i], sm = sign_mask(NQ);
  int g = 0;
#pragma unroll
  for (int q = 0; q < NQ; q++)
#pragma unroll
    for (int k = 0; k < 2; k++, g++) nb[(size_t)g * C + i] = (uint32_t)find_sym(T, apply(t, NQ, k, q, 0) & ~sm);
#pragma unroll
  for (int x = 0; x < NQ; x++)
#pragma unroll
    for (int y = 0; y < NQ; y++)
      if (x != y) { nb[(size_t)g * C + i] = (uint32_t)find_sym(T, apply(t, NQ, 5, x, y) & ~sm); g++; }
}

struct BfsArgs {
  const uint64_t *key;
  const uint32_t *nb;
  const uint64_t *front;       // per matrix, the sign vectors at distance d - 1
  uint64_t *next;              // those at distance d
  uint64_t *seen;
  ulonglong2 *planes;
  uint8_t *dmin;
  unsigned long long *cnt;     // elements per distance
  int d;
};

// One level of the search, one thread per matrix: the sign vectors at distance d are those that a gate brings from a
// matrix's sign vectors at distance d - 1, a set of 2^(2n) bits XOR-shifted by the gate's sign vector, less those seen
// before.  Each (element, gate) pair is one bit of a 64-bit operation and each (matrix, gate) pair one gather from an
// 11.6 MB array, where a hash table of whole tableaux took a probe of a random 128-byte line per pair: the 3-qubit
// group (1.95 billion pairs) took 164 ms, all its levels here 0.84, numbering and neighbours 0.4 more.
template <int NQ> __global__ __launch_bounds__(256) void k_bfs(BfsArgs a) {
  constexpr uint32_t C = (uint32_t)Num<NQ>::matrices();
  constexpr int M = 2 * NQ, RB = M + 1;
  if (!a.cnt[a.d - 1]) return;                       // the level before is empty
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  uint64_t acc = 0, nx = 0;
  if (i < C) {
    const uint64_t t = a.key[i];
    // column c of the matrix (x_0.. then z_0..), row r in bit r
    uint32_t col[M];
#pragma unroll
    for (int c = 0; c < M; c++) {
      col[c] = 0;
#pragma unroll
      for (int r = 0; r < M; r++) col[c] |= (uint32_t)((t >> (r * RB + c)) & 1) << r;
    }
    const uint64_t own = a.front[i];
    int g = 0;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
      const uint32_t x = col[q], z = col[NQ + q];
      if (own) acc |= Num<NQ>::shift(own, z) | Num<NQ>::shift(own, x);                       // X, Z
      const uint64_t h = a.front[a.nb[(size_t)g++ * C + i]];
      if (h) acc |= Num<NQ>::shift(h, x & z);                                                // H
      const uint64_t p = a.front[a.nb[(size_t)g++ * C + i]];
      if (p) acc |= Num<NQ>::shift(p, x & ~z) | Num<NQ>::shift(p, x & z);                     // S, Sdg
    }
#pragma unroll
    for (int x = 0; x < NQ; x++)
#pragma unroll
      for (int y = 0; y < NQ; y++)
        if (x != y) {
          const uint64_t f = a.front[a.nb[(size_t)g++ * C + i]];
          if (f) acc |= Num<NQ>::shift(f, col[x] & col[NQ + y] & ~(col[y] ^ col[NQ + x]));    // CX x -> y
        }
    const uint64_t s = a.seen[i];
    nx = acc & ~s;
    a.next[i] = nx;
    if (nx) {
      a.seen[i] = s | nx;
      if (!s) a.dmin[i] = (uint8_t)a.d;
      ulonglong2 p = a.planes[2 * i], q = a.planes[2 * i + 1];
      if (a.d & 1) p.x |= nx;
      if (a.d & 2) p.y |= nx;
      if (a.d & 4) q.x |= nx;
      if (a.d & 8) q.y |= nx;
      a.planes[2 * i] = p;
      a.planes[2 * i + 1] = q;
    }
  }
  __shared__ uint32_t ws[4];
  const uint32_t c = gsum<64>((uint32_t)__popcll(nx));
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    const uint32_t tot = ws[0] + ws[1] + ws[2] + ws[3];
    if (tot) atomicAdd(&a.cnt[a.d], (unsigned long long)tot);
  }
}

__global__ void k_fill_u64(unsigned long long *p, long long n) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) p[i] = 0;
}
// the identity at distance 0
__global__ void k_root(Table T, uint64_t id, uint64_t *front, uint64_t *seen, unsigned long long *cnt) {
  if (blockIdx.x || threadIdx.x) return;
  const int i = find_sym(T, id);
  front[i] = 1;
  seen[i] = 1;
  cnt[0] = 1;
}

// ---- words.  A tableau's X images and its Z images are two words of n rows each; a gate acts on all rows of a word
// at once.  A letter's gate is packed as its qubits and one flag per term of the update:
enum { W_HS = 8, W_SDG, W_Z, W_X, W_CX, W_H, W_SZ };     // bits 0-3: a, 4-7: b; H or S, Sdg, Z, X, CX, H, S or Sdg
static uint32_t pack_gate(int k, int a, int b) {
  uint32_t f = (uint32_t)a | (uint32_t)b << 4;
  if (k == 0) f |= 1u << W_HS | 1u << W_H;
  else if (k == 1) f |= 1u << W_HS | 1u << W_SZ;
  else if (k == 2) f |= 1u << W_SDG | 1u << W_SZ;
  else if (k == 3) f |= 1u << W_X;
  else if (k == 4) f |= 1u << W_Z;
  else f |= 1u << W_CX;
  return f;
}
struct WordGates { uint32_t g[32]; };
static WordGates word_gates(const Gates &G) {
  WordGates w{};
  for (int i = 0; i < G.ng; i++) w.g[i] = pack_gate(G.k[i], G.a[i], G.b[i]);
  return w;
}
template <int NQ> __device__ __forceinline__ uint32_t apply_rows(uint32_t w, uint32_t g) {
  constexpr uint32_t M = NQ == 1 ? 1u : NQ == 2 ? 1u | 1u << 5 : 1u | 1u << 7 | 1u << 14;      // bit 0 of every row
  auto on = [&](int bit) -> uint32_t { return (uint32_t)__builtin_amdgcn_sbfe((int)g, (unsigned)bit, 1u); };
  const uint32_t a = g & 15u, b = (g >> 4) & 15u;
  const uint32_t xa = w >> a & M, za = w >> (NQ + a) & M, xb = w >> b & M, zb = w >> (NQ + b) & M;
  const uint32_t h = (xa ^ za) & on(W_H), xc = xa & on(W_CX);
  const uint32_t sign = (xa & ((za & on(W_HS)) | (~za & on(W_SDG)) | on(W_Z))) | (za & on(W_X)) | (xc & zb & ~(xb ^ za));
  return w ^ (sign << (2 * NQ)) ^ (h << a) ^ ((h ^ (xa & on(W_SZ)) ^ (zb & on(W_CX))) << (NQ + a)) ^ (xc << b);
}

// distances of words (letters are gate-set indices, applied in order; src/clifford.cu:207-210), one lane per word.  A
// wave's letters are one range of memory: it is read as whole dwords into LDS, where the lanes pick their letters, when
// it fits and the lanes' ranges lie in it; otherwise each lane reads its letters from global memory.
// What bounded this: a serial chain per lane of byte loads from global memory, each letter's gate read from a per-lane
// index into the kernel arguments and applied row by row in six divergent ways, then a second kernel for the look-ups:
// 96 + 5 us for 1e5 words of 5 to 40 letters, 19 us here.
constexpr int WORD_SPAN = 4096;        // bytes of letters per wave in LDS
template <int NQ>
__global__ __launch_bounds__(256) void k_query(Table T, WordGates G, const uint8_t *letters, const long long *offs, long long nq,
                                               int *out) {
  constexpr int HB = NQ * (2 * NQ + 1);      // bits of a word of n rows
  __shared__ uint32_t stage[4][WORD_SPAN / 4], gate[32];
  if (threadIdx.x < 32) gate[threadIdx.x] = G.g[threadIdx.x];
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const uint64_t id = identity(NQ);
  for (long long q0 = wave_index() * 64; q0 < nq; q0 += (long long)gridDim.x * 256) {
    const long long q = q0 + lane, last = q0 + 64 < nq ? q0 + 64 : nq;
    const long long beg = q < nq ? offs[q] : 0, end = q < nq ? offs[q + 1] : 0;
    const long long lo = offs[q0], hi = offs[last];
    // LDS byte i holds the letter at address base + i (base: lo rounded down to a dword)
    const uintptr_t first = (uintptr_t)letters + (uintptr_t)lo, base = first & ~(uintptr_t)3, stop = (uintptr_t)letters + (uintptr_t)hi;
    const bool staged = hi - lo <= WORD_SPAN - 4 && hi >= lo &&
                        __ballot(q < nq && beg < end && (beg < lo || end > hi)) == 0;
    uint32_t x = (uint32_t)(id & ((1ull << HB) - 1)), z = (uint32_t)(id >> HB);
    if (staged) {
      uint8_t *const s8 = (uint8_t *)stage[wv];
      const uintptr_t d0 = (first + 3) & ~(uintptr_t)3, d1 = stop & ~(uintptr_t)3;      // whole dwords [d0, d1)
      for (uintptr_t p = d0 + 4 * lane; p < d1; p += 256) stage[wv][(p - base) >> 2] = *(const uint32_t *)p;
      // the bytes before and behind them, at most three each
      if (lane < 3 && first + lane < d0 && first + lane < stop) s8[first + lane - base] = *(const uint8_t *)(first + lane);
      if (lane >= 4 && lane < 7 && d1 >= d0 && d1 + (lane - 4) < stop) s8[d1 + (lane - 4) - base] = *(const uint8_t *)(d1 + (lane - 4));
      __builtin_amdgcn_wave_barrier();
      const int off = (int)((uintptr_t)letters + (uintptr_t)beg - base), len = beg < end ? (int)(end - beg) : 0;
      for (int j = 0; j < len; j++) {
        const uint32_t g = gate[s8[off + j] & 31];
        x = apply_rows<NQ>(x, g);
        z = apply_rows<NQ>(z, g);
      }
      __builtin_amdgcn_wave_barrier();
    } else {
      for (long long j = beg; j < end; j++) {
        const uint32_t g = gate[letters[j] & 31];
        x = apply_rows<NQ>(x, g);
        z = apply_rows<NQ>(z, g);
      }
    }
    if (q < nq) out[q] = find1(T, (uint64_t)x | (uint64_t)z << HB);
  }
}
static void launch_query(const Table &T, const Gates &G, const uint8_t *letters, const long long *offs, long long nq, int *out,
                         hipStream_t s) {
  const dim3 g((unsigned)std::min<long long>((nq + 255) / 256 + (nq == 0), 4096)), b(256);
  const WordGates w = word_gates(G);
  if (G.n == 1) hipLaunchKernelGGL(k_query<1>, g, b, 0, s, T, w, letters, offs, nq, out);
  else if (G.n == 2) hipLaunchKernelGGL(k_query<2>, g, b, 0, s, T, w, letters, offs, nq, out);
  else hipLaunchKernelGGL(k_query<3>, g, b, 0, s, T, w, letters, offs, nq, out);
}

// optimal words: one wave per query; each step, lane g tests the predecessor through gate g (its distance
// must be one less) and the first such gate in gate order is taken (src/clifford.cu:354-372)
__global__ __launch_bounds__(64) void k_readback(Gates G, Table T, const uint64_t *q, long long nq, int maxlen,
                                                 uint8_t *words, int *lens) {
  const int lane = threadIdx.x;
  for (long long i = blockIdx.x; i < nq; i += gridDim.x) {
    uint64_t X = q[i];
    const int d = find1(T, X);
    if (d < 0 || d > maxlen) { if (lane == 0) lens[i] = -1; continue; }
    if (lane == 0) lens[i] = d;
    for (int s = d; s > 0; s--) {
      uint64_t pre = 0;
      bool ok = false;
      if (lane < G.ng) {
        pre = apply(X, G.n, inv_kind(G.k[lane]), G.a[lane], G.b[lane]);
        ok = find1(T, pre) == s - 1;
      }
      const uint64_t bal = __ballot(ok);
      const int g = bal ? __ffsll((long long)bal) - 1 : -1;
      if (g < 0) { if (lane == 0) lens[i] = -1; break; }
      X = __shfl(pre, g, 64);
      if (lane == 0) words[i * maxlen + (s - 1)] = (uint8_t)g;
    }
  }
}

// seeded uniform elements: splitmix64 numbers of elements in the order of their tableaux
template <int NQ> __global__ __launch_bounds__(256) void k_sample(unsigned long long seed, long long n, uint64_t *out) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
    uint64_t z = seed + (uint64_t)(i + 1) * 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    z ^= z >> 31;
    out[i] = Num<NQ>::element(z % (uint64_t)Num<NQ>::ORDER);
  }
}

// order-independent digest: sum over entries of hmix-free mix of (tableau * 64 + distance), and the count
__global__ __launch_bounds__(256) void k_digest(Table T, const uint64_t *key, long long count, unsigned long long *out) {
  unsigned long long s = 0, c = 0;
  const int n = T.n, ns = 1 << (2 * n);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (long long)gridDim.x * blockDim.x) {
    const uint64_t t = key[i];
    const ulonglong2 p = T.planes[2 * i], q = T.planes[2 * i + 1];
    for (int v = 0; v < ns; v++) {
      uint64_t w = t;
      for (int r = 0; r < 2 * n; r++) w |= (uint64_t)((v >> r) & 1) << (r * (2 * n + 1) + 2 * n);
      uint64_t x = w * 64 + (uint64_t)plane_dist(p, q, (uint32_t)v);
      x ^= x >> 33; x *= 0xff51afd7ed558ccdull; x ^= x >> 33;
      x *= 0xc4ceb9fe1a85ec53ull; x ^= x >> 33; s += x; c++;
    }
  }
  for (int m = 1; m < 64; m <<= 1) { s += __shfl_xor(s, m, 64); c += __shfl_xor(c, m, 64); }
  if ((threadIdx.x & 63) == 0) { atomicAdd(&out[0], s); atomicAdd(&out[1], c); }
}

static thread_local std::string g_err;

#include "cliffopt_kernels.h"

}  // namespace chz_cl

namespace chz_cl {
constexpr long long kQueryWords = 1ll << 20;      // most words of one chz_cliff_query_words_noalloc call
}

struct chz_cliff {
  int n = 0, device = 0;
  chz_cl::Gates G{};
  chz_cl::Table T{};
  void *block = nullptr;               // the table's arrays, one block
  uint64_t *key = nullptr;             // sign-free tableaux of the matrices
  long long count = 0;                 // matrices
  std::vector<long> levels;
  hipStream_t stream = nullptr;
  double build_ms = 0;
};

#define CLCHK(x)                                                                         \
  do {                                                                                   \
    hipError_t e_ = (x);                                                                 \
    if (e_ != hipSuccess) { chz_cl::g_err = std::string("HIP error: ") + hipGetErrorString(e_); return 5; } \
  } while (0)

extern "C" {

const char *chz_cliff_last_error(void) { return chz_cl::g_err.c_str(); }

}  // extern "C"

// the table of c (its stream and n set); 0, 4 or 5
template <int NQ> static int cliff_fill(chz_cliff *c) {
  using namespace chz_cl;
  constexpr long long C = Num<NQ>::matrices();
  constexpr int MAXD = NQ == 1 ? 3 : NQ == 2 ? 9 : 13;    // the group's largest distance (its order is checked below)
  static_assert(MAXD < 16, "four planes");
  long long slots = 64;
  while (slots < 2 * C) slots <<= 1;
  auto up = [](size_t b) { return (b + 255) & ~(size_t)255; };
  // [slots | planes | smallest distances | keys], and for the build [seen | two frontiers | counts | neighbours]
  const size_t o_pl = up(slots * 8), o_min = o_pl + up(C * 32), o_key = o_min + up(C), bytes = o_key + up(C * 8);
  const size_t w_f0 = up(C * 8), w_f1 = 2 * w_f0, w_cnt = 3 * w_f0, w_nb = w_cnt + 256, wbytes = w_nb + up((size_t)sym_gates(NQ) * C * 4);
  uint8_t *work = nullptr;
  CLCHK(cl_malloc(&c->block, bytes));
  CLCHK(cl_malloc((void **)&work, wbytes));
  struct Guard { uint8_t *p; ~Guard() { (void)cl_free(p); } } guard{work};     // (hipFree waits for the device)
  uint8_t *blk = (uint8_t *)c->block;
  c->count = C;
  c->key = (uint64_t *)(blk + o_key);
  c->T = Table{(unsigned long long *)blk, (uint32_t)(slots - 1), (const ulonglong2 *)(blk + o_pl), blk + o_min, NQ};
  uint64_t *seen = (uint64_t *)work, *front[2] = {(uint64_t *)(work + w_f0), (uint64_t *)(work + w_f1)};
  unsigned long long *cnt = (unsigned long long *)(work + w_cnt);
  uint32_t *nb = (uint32_t *)(work + w_nb);
  hipEvent_t e0, e1;
  CLCHK(hipEventCreate(&e0));
  CLCHK(hipEventCreate(&e1));
  CLCHK(hipEventRecord(e0, c->stream));
  const dim3 grid((unsigned)((C + 255) / 256)), blockd(256);
  hipLaunchKernelGGL(k_fill_u64, dim3(4096), blockd, 0, c->stream, (unsigned long long *)blk, (long long)(o_key / 8));
  hipLaunchKernelGGL(k_fill_u64, dim3(4096), blockd, 0, c->stream, (unsigned long long *)work, (long long)(w_nb / 8));
  hipLaunchKernelGGL(k_matrices<NQ>, grid, blockd, 0, c->stream, c->key, c->T.slot, c->T.smask);
  hipLaunchKernelGGL(k_neighbours<NQ>, grid, blockd, 0, c->stream, c->T, c->key, nb);
  hipLaunchKernelGGL(k_root, dim3(1), dim3(64), 0, c->stream, c->T, identity(NQ), front[0], seen, cnt);
  // every level is queued at once
  for (int d = 1; d <= MAXD; d++) {
    const BfsArgs a{c->key, nb, front[(d - 1) & 1], front[d & 1], seen, (ulonglong2 *)(blk + o_pl), blk + o_min, cnt, d};
    hipLaunchKernelGGL(k_bfs<NQ>, grid, blockd, 0, c->stream, a);
  }
  CLCHK(hipGetLastError());
  unsigned long long h[MAXD + 1];
  CLCHK(hipMemcpyAsync(h, cnt, sizeof h, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipEventRecord(e1, c->stream));
  CLCHK(hipStreamSynchronize(c->stream));
  float ms = 0;
  CLCHK(hipEventElapsedTime(&ms, e0, e1));
  c->build_ms = ms;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  long long total = 0;
  for (int d = 0; d <= MAXD && h[d]; d++) {
    c->levels.push_back((long)h[d]);
    total += (long long)h[d];
  }
  if (total != Num<NQ>::ORDER) { g_err = "group order mismatch"; return 4; }   // src/clifford.cu:279-280
  return 0;
}

extern "C" {

int chz_cliff_build(int n, int device, chz_cliff **out) {
  chz::RelaxedCapture relaxed;
  *out = nullptr;
  if (n < 1 || n > 3) { chz_cl::g_err = "n must be 1..3"; return 3; }
  CLCHK(hipSetDevice(device));
  chz_cliff *c = new chz_cliff();
  c->n = n;
  c->device = device;
  c->G = chz_cl::gate_set(n);
  if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    chz_cl::g_err = "HIP error: no stream";
    delete c;
    return 5;
  }
  const int rc = n == 1 ? cliff_fill<1>(c) : n == 2 ? cliff_fill<2>(c) : cliff_fill<3>(c);
  if (rc == 5) { chz_cliff_free(c); return 5; }
  *out = c;
  return rc;
}

int chz_cliff_levels(const chz_cliff *c, long *counts, int maxd) {
  const int nl = (int)c->levels.size();
  for (int i = 0; i < nl && i < maxd; i++) counts[i] = c->levels[i];
  return nl;
}

int chz_cliff_num_gates(const chz_cliff *c) { return c->G.ng; }

double chz_cliff_build_ms(const chz_cliff *c) { return c->build_ms; }

int chz_cliff_digest(const chz_cliff *c, uint64_t *digest, long long *entries) {
  unsigned long long *d = nullptr, h[2] = {0, 0};
  CLCHK(hipSetDevice(c->device));
  CLCHK(cl_malloc((void **)&d, 16));
  CLCHK(hipMemsetAsync(d, 0, 16, c->stream));
  hipLaunchKernelGGL(chz_cl::k_digest, dim3(2048), dim3(256), 0, c->stream, c->T, c->key, c->count, d);
  CLCHK(hipMemcpyAsync(h, d, 16, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipStreamSynchronize(c->stream));
  (void)cl_free(d);
  *digest = h[0];
  *entries = (long long)h[1];
  return 0;
}

// count uniformly random group elements (tableaux), seeded: uniform numbers in the order of the tableaux, so that
// samples do not depend on anything but the seed
int chz_cliff_sample(chz_cliff *c, uint64_t seed, long long count, uint64_t *tab) {
  CLCHK(hipSetDevice(c->device));
  uint64_t *d = nullptr;
  CLCHK(cl_malloc((void **)&d, std::max<long long>(count, 1) * 8));
  const dim3 g((unsigned)std::min<long long>((count + 255) / 256 + 1, 4096)), b(256);
  if (c->n == 1) hipLaunchKernelGGL(chz_cl::k_sample<1>, g, b, 0, c->stream, (unsigned long long)seed, count, d);
  else if (c->n == 2) hipLaunchKernelGGL(chz_cl::k_sample<2>, g, b, 0, c->stream, (unsigned long long)seed, count, d);
  else hipLaunchKernelGGL(chz_cl::k_sample<3>, g, b, 0, c->stream, (unsigned long long)seed, count, d);
  CLCHK(hipMemcpyAsync(tab, d, count * 8, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipStreamSynchronize(c->stream));
  (void)cl_free(d);
  return 0;
}

// distances of nq words: letters[offs[i] .. offs[i+1]) are gate-set indices applied in order.
// ms (may be NULL) receives the device time of the word and lookup kernels.
int chz_cliff_query_words(chz_cliff *c, const uint8_t *letters, const long long *offs, long long nq, int *dist,
                          double *ms) {
  chz::RelaxedCapture relaxed;
  CLCHK(hipSetDevice(c->device));
  const long long nl = offs[nq];
  uint8_t *dl = nullptr;
  long long *doff = nullptr;
  int *dd = nullptr;
  CLCHK(cl_malloc((void **)&dl, std::max<long long>(nl, 1)));
  CLCHK(cl_malloc((void **)&doff, (nq + 1) * 8));
  CLCHK(cl_malloc((void **)&dd, std::max<long long>(nq, 1) * 4));
  CLCHK(hipMemcpyAsync(dl, letters, nl, hipMemcpyHostToDevice, c->stream));
  CLCHK(hipMemcpyAsync(doff, offs, (nq + 1) * 8, hipMemcpyHostToDevice, c->stream));
  hipEvent_t e0, e1;
  CLCHK(hipEventCreate(&e0));
  CLCHK(hipEventCreate(&e1));
  CLCHK(hipEventRecord(e0, c->stream));
  chz_cl::launch_query(c->T, c->G, dl, doff, nq, dd, c->stream);
  CLCHK(hipEventRecord(e1, c->stream));
  CLCHK(hipMemcpyAsync(dist, dd, nq * 4, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipStreamSynchronize(c->stream));
  float t = 0;
  CLCHK(hipEventElapsedTime(&t, e0, e1));
  if (ms) *ms = t;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  (void)cl_free(dl);
  (void)cl_free(doff);
  (void)cl_free(dd);
  return 0;
}

// chz_cliff_query_words with device buffers and no allocation, at most kQueryWords words per call; the kernel goes on
// `stream` (NULL: the table's own stream, synchronised before returning).
int chz_cliff_query_words_noalloc(chz_cliff *c, const uint8_t *d_letters, const long long *d_offs, long long nq,
                                  int *d_dist, void *stream) {
  if (nq < 0 || (nq > 0 && (!d_letters || !d_offs || !d_dist))) { chz_cl::g_err = "bad arguments"; return 3; }
  if (nq > chz_cl::kQueryWords) {
    chz_cl::g_err = "chz_cliff_query_words_noalloc: " + std::to_string(nq) + " words exceed the scratch capacity of " +
                    std::to_string(chz_cl::kQueryWords);
    return 4;
  }
  if (nq == 0) return 0;
  chz::RelaxedCapture relaxed;
  CLCHK(hipSetDevice(c->device));
  hipStream_t st = stream ? (hipStream_t)stream : c->stream;
  chz_cl::launch_query(c->T, c->G, d_letters, d_offs, nq, d_dist, st);
  CLCHK(hipGetLastError());
  if (!stream) CLCHK(hipStreamSynchronize(st));
  return 0;
}

// tableau of one word (host arithmetic, same algebra as the device)
uint64_t chz_cliff_word_tableau(const chz_cliff *c, const uint8_t *letters, int len) {
  uint64_t T = chz_cl::identity(c->n);
  for (int i = 0; i < len; i++) {
    const int g = letters[i];
    T = chz_cl::apply(T, c->n, c->G.k[g], c->G.a[g], c->G.b[g]);
  }
  return T;
}

// optimal words of nq tableaux (gate-set indices, <= maxlen each); lens[i] = length or -1
int chz_cliff_readback(chz_cliff *c, const uint64_t *tab, long long nq, int maxlen, uint8_t *words, int *lens) {
  chz::RelaxedCapture relaxed;
  CLCHK(hipSetDevice(c->device));
  uint64_t *dt = nullptr;
  uint8_t *dw = nullptr;
  int *dlen = nullptr;
  CLCHK(cl_malloc((void **)&dt, std::max<long long>(nq, 1) * 8));
  CLCHK(cl_malloc((void **)&dw, std::max<long long>(nq * maxlen, 1)));
  CLCHK(cl_malloc((void **)&dlen, std::max<long long>(nq, 1) * 4));
  CLCHK(hipMemcpyAsync(dt, tab, nq * 8, hipMemcpyHostToDevice, c->stream));
  hipLaunchKernelGGL(chz_cl::k_readback, dim3((unsigned)std::min<long long>(std::max<long long>(nq, 1), 8192)),
                     dim3(64), 0, c->stream, c->G, c->T, dt, nq, maxlen, dw, dlen);
  CLCHK(hipMemcpyAsync(words, dw, nq * maxlen, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipMemcpyAsync(lens, dlen, nq * 4, hipMemcpyDeviceToHost, c->stream));
  CLCHK(hipStreamSynchronize(c->stream));
  (void)cl_free(dt);
  (void)cl_free(dw);
  (void)cl_free(dlen);
  return 0;
}

void chz_cliff_free(chz_cliff *c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->block) (void)cl_free(c->block);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

}  // extern "C"

#include "cliffopt.h"
