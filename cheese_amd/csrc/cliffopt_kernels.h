// Device side of the T-placement beam search (`cliffopt`, src/clifford.cu:168-206): tableau composition and
// inversion, the placements of a T gate, one beam step with an in-block top-B selection, and the final segment
// lookup.  Included by clifford.hip inside namespace chz_cl, after the tableau and table definitions.
//
// A T gate on qubit q commutes with every Clifford K with K Z_q' K^-1 = +-Z_q, so T_q can be replaced by
// K T'_q' K^-1 (T' with its dagger flipped for the minus sign) at the cost of a global phase; segment j of the
// circuit then becomes K_{j+1}^-1 D_j K_j.  The beam search picks K for every T gate so that the summed optimal
// segment lengths (read from the Clifford table) are small; T = Tdg S and Tdg = T Sdg exactly, so a T may also
// flip its dagger, moving an S (Sdg) into the segment before it.

__host__ __device__ inline uint32_t trow(uint64_t T, int n, int i) {
  const int rb = 2 * n + 1;
  return (uint32_t)((T >> (i * rb)) & ((1ull << rb) - 1));
}
__host__ __device__ inline uint64_t tset(uint64_t T, int n, int i, uint32_t r) {
  const int rb = 2 * n + 1;
  const uint64_t m = ((1ull << rb) - 1) << (i * rb);
  return (T & ~m) | ((uint64_t)r << (i * rb));
}

// the Clifford's image of the Hermitian Pauli i^(x.z) X^x Z^z, as a row: the product of the images of its X and
// then Z factors, the power of i tracked through (X^a Z^b)(X^c Z^d) = (-1)^(b.c) X^(a^c) Z^(b^d)
__host__ __device__ inline uint32_t timage(uint64_t T, int n, uint32_t x, uint32_t z) {
  const uint32_t nm = (1u << n) - 1;
  int k = __builtin_popcount(x & z);
  uint32_t ax = 0, az = 0;
  for (int g = 0; g < 2 * n; g++) {
    const bool on = g < n ? ((x >> g) & 1) : ((z >> (g - n)) & 1);
    if (!on) continue;
    const uint32_t w = trow(T, n, g), bx = w & nm, bz = (w >> n) & nm, r = (w >> (2 * n)) & 1;
    k += 2 * (int)r + __builtin_popcount(bx & bz) + 2 * __builtin_popcount(az & bx);
    ax ^= bx;
    az ^= bz;
  }
  const uint32_t sign = (uint32_t)(((k - __builtin_popcount(ax & az)) & 3) >> 1);
  return ax | (az << n) | (sign << (2 * n));
}

// A then B: row i of the product is B's image of A's row i, its sign carried
__host__ __device__ inline uint64_t tcompose(uint64_t A, uint64_t B, int n) {
  const uint32_t nm = (1u << n) - 1;
  uint64_t C = 0;
  for (int i = 0; i < 2 * n; i++) {
    const uint32_t w = trow(A, n, i);
    C = tset(C, n, i, timage(B, n, w & nm, (w >> n) & nm) ^ (((w >> (2 * n)) & 1) << (2 * n)));
  }
  return C;
}

// the inverse: its symplectic part is Omega S^T Omega (S the tableau's bit matrix), and the sign of row i is the one
// with which the Clifford maps that row's Pauli back onto generator i
__host__ __device__ inline uint64_t tinverse(uint64_t C, int n) {
  const int m = 2 * n;
  const uint32_t nm = (1u << n) - 1;
  uint64_t D = 0;
  for (int i = 0; i < m; i++) {
    const int wi = (i + n) % m;
    uint32_t v = 0;
    for (int j = 0; j < m; j++) {
      const uint32_t sr = trow(C, n, (j + n) % m);
      v |= (((sr & nm) | (((sr >> n) & nm) << n)) >> wi & 1) << j;
    }
    const uint32_t x = v & nm, z = v >> n;
    D = tset(D, n, i, x | (z << n) | (((timage(C, n, x, z) >> (2 * n)) & 1) << (2 * n)));
  }
  return D;
}

struct Cand { uint64_t K, Kinv; int qp, neg; };

// the qubit q' with K Z_q' K^-1 = +-Z_q, -1 when K is no placement for a T on qubit q
__host__ __device__ inline int placement_of(uint64_t K, int n, int q) {
  for (int qp = 0; qp < n; qp++)
    if ((trow(K, n, n + qp) & ((1u << (2 * n)) - 1)) == 1u << (n + q)) return qp;
  return -1;
}
__host__ __device__ inline Cand make_cand(uint64_t K, int n, int q) {
  const int qp = placement_of(K, n, q);
  return Cand{K, tinverse(K, n), qp, (int)((trow(K, n, n + qp) >> (2 * n)) & 1)};
}

// Placements depend on the Z images alone, which lead an element's number: Z images number z (signed: of all signed
// ones) hold placements or none, and the placements in the order of their tableaux are the elements z * X_ALL + x of
// the flagged z.
template <int NQ> struct FlagZ {          // unsigned Z images
  int q;
  __device__ bool operator()(long long z) const { return placement_of(Num<NQ>::matrix((uint32_t)z * Num<NQ>::X_SYM), NQ, q) >= 0; }
};
template <int NQ> struct FlagZs {         // signed Z images
  int q;
  __device__ bool operator()(long long z) const { return placement_of(Num<NQ>::element((uint64_t)z * Num<NQ>::X_ALL), NQ, q) >= 0; }
};
__global__ void k_invert(const uint32_t *list, const unsigned long long *n, uint32_t *out) {
  const long long cnt = (long long)*n;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < cnt; i += (long long)gridDim.x * blockDim.x)
    out[list[i]] = (uint32_t)i;
}

// a placement's matrix: its number, its inverse (as a sign-free tableau's) and q'
struct PlaceMat { uint64_t K, Kinv; uint32_t num; int qp; };
template <int NQ> __global__ __launch_bounds__(256) void k_place(const uint32_t *zlist, long long nm, int q, PlaceMat *out) {
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < nm; i += (long long)gridDim.x * 256) {
    const uint32_t m = zlist[i / Num<NQ>::X_SYM] * Num<NQ>::X_SYM + (uint32_t)(i % Num<NQ>::X_SYM);
    const uint64_t K = Num<NQ>::matrix(m);
    out[i] = PlaceMat{K, tinverse(K, NQ), m, placement_of(K, NQ, q)};
  }
}

// T = Tdg S: a flipped placement's inverse takes an S (Sdg when the placed T is a dagger) after it
__host__ __device__ inline uint64_t flipped_inv(const Cand &c, int dagger, int n) {
  return apply(c.Kinv, n, dagger ? 2 : 1, c.qp, 0);
}

constexpr int TOPK = 256;   // largest beam

// the block's B smallest values among best[0..256) and vals[0..256): bitonic sort of the 512 in LDS
__device__ inline void merge_topk(unsigned long long *best) {
  const int tid = threadIdx.x;
  for (int size = 2; size <= 512; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();
      for (int e = tid; e < 256; e += blockDim.x) {   // 256 compare-exchanges per stage
        const int lo = (e / stride) * stride * 2 + (e % stride), hi = lo + stride;
        const bool up = (lo & size) == 0;
        const unsigned long long a = best[lo], b = best[hi];
        if ((a > b) == up) { best[lo] = b; best[hi] = a; }
      }
    }
  __syncthreads();
}

struct BeamArgs {
  Table T;
  const uint64_t *left;     // per state: the placement kept by the step before and then this T gate's preceding segment
  const int *bcost;         // per state: its summed segment lengths
  int nb, minb;             // states, the smallest of bcost
  const PlaceMat *pm;       // placements' matrices
  long long nm;
  const uint32_t *zpos;     // signed Z images -> their place among the flagged
  uint8_t *low;             // per row: a lower bound on its items' cost, above minb (255: that or more)
  unsigned int *hist;       // rows per bound
  int dg;                   // this T gate's dagger before any flip
  int B;
  unsigned long long *out;  // per block: its B smallest (cost << 40 | state << 32 | candidate << 1 | flip)
};

// The placements of one beam step (src/clifford.cu:190-201) that share a matrix differ by signs, and so do the segments
// they leave: their products range over the sign vectors of one matrix.  So a row (state, placement matrix, flip) of
// 2^(2n) items is bounded from below by that matrix's smallest distance (k_beam_low), the rows' bounds give a cost that
// at least B items do not exceed, and only rows whose bound does not exceed it are looked at item by item (k_beam).
// At 3 qubits a step of 16 states has 2.2 million rows for 141 million items, each of which took a composition and a probe
// of a 1.07 GB table: 5 ms a step, against 0.05 (bounds) and 0.04 (items) here.
template <int NQ> __global__ __launch_bounds__(256) void k_beam_low(BeamArgs a) {
  __shared__ unsigned int h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const long long rows = (long long)a.nb * a.nm * 2;
  const uint64_t sm = sign_mask(NQ);
  for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < rows; i += (long long)gridDim.x * 256) {
    const int b = (int)(i / (a.nm * 2)), f = (int)(i & 1);
    const PlaceMat pm = a.pm[(i % (a.nm * 2)) >> 1];
    const uint64_t kinv = f ? apply(pm.Kinv, NQ, 1, pm.qp, 0) : pm.Kinv;
    const int m = find_sym(a.T, tcompose(a.left[b], kinv, NQ) & ~sm);
    const int lo = a.bcost[b] - a.minb + (m < 0 ? 0 : a.T.dmin[m]), r = lo < 255 ? lo : 255;
    a.low[i] = (uint8_t)r;
    atomicAdd(&h[r], 1u);
  }
  __syncthreads();
  if (h[threadIdx.x]) atomicAdd(&a.hist[threadIdx.x], h[threadIdx.x]);
}

// the step's B smallest items, each block keeping those of its contiguous range of rows in LDS
template <int NQ> __global__ __launch_bounds__(256) void k_beam(BeamArgs a) {
  __shared__ unsigned long long best[512];
  __shared__ uint32_t queue[256 + 4];
  __shared__ unsigned int nq, thr;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  best[tid] = ~0ull;
  best[256 + tid] = ~0ull;
  if (tid == 0) {
    unsigned int c = 0, t = 0;         // the smallest bound that at least B rows do not exceed (255: every row)
    for (; t < 255; t++) if ((c += a.hist[t]) >= (unsigned)a.B) break;
    thr = t;
    nq = 0;
  }
  __syncthreads();
  const long long rows = (long long)a.nb * a.nm * 2, per = (rows + gridDim.x - 1) / gridDim.x;
  const long long lo = (long long)blockIdx.x * per, hi = lo + per < rows ? lo + per : rows;
  const unsigned int limit = thr;
  for (long long base = lo; base < hi; base += 256) {
    const long long i = base + tid;
    if (i < hi && a.low[i] <= limit) queue[atomicAdd(&nq, 1u)] = (uint32_t)(i - lo);
    __syncthreads();
    const bool last = base + 256 >= hi;
    unsigned int left = nq;
    // four rows at a time, one per wave (fewer than four wait for the next rows)
    while (left >= 4 || (last && left)) {
      unsigned long long v = ~0ull;
      if ((unsigned)w < left) {
        const long long row = lo + queue[left - 1 - w];
        const int b = (int)(row / (a.nm * 2)), f = (int)(row & 1);
        // the row's smallest possible value against the block's B-th smallest so far
        const unsigned long long least =
            (unsigned long long)(a.low[row] < 255 ? a.minb + a.low[row] : a.bcost[b]) << 40 | (unsigned long long)b << 32;
        if (least < best[a.B - 1] && lane < 1 << (2 * NQ)) {
          const PlaceMat pm = a.pm[(row % (a.nm * 2)) >> 1];
          uint64_t K = pm.K;
#pragma unroll
          for (int r = 0; r < 2 * NQ; r++) K |= (uint64_t)((lane >> r) & 1) << (r * (2 * NQ + 1) + 2 * NQ);
          const Cand cd{K, tinverse(K, NQ), pm.qp, (lane >> (NQ + pm.qp)) & 1};
          const int d = find1(a.T, tcompose(a.left[b], f ? flipped_inv(cd, a.dg ^ cd.neg, NQ) : cd.Kinv, NQ));
          const unsigned long long cost = (unsigned long long)(a.bcost[b] + (d < 0 ? 999 : d));
          const uint64_t e = Num<NQ>::signed_number(pm.num, (uint32_t)lane);
          const uint64_t c = (uint64_t)a.zpos[e / Num<NQ>::X_ALL] * Num<NQ>::X_ALL + e % Num<NQ>::X_ALL;
          v = (cost << 40) | ((unsigned long long)b << 32) | (c << 1 | (unsigned)f);
        }
      }
      left -= left < 4 ? left : 4;
      // merge only when some new value beats the block's current B-th smallest
      if (__syncthreads_or(v < best[a.B - 1])) {
        best[256 + tid] = v;
        merge_topk(best);
      }
    }
    __syncthreads();
    if (tid == 0) nq = left;
    __syncthreads();
  }
  for (int j = tid; j < a.B; j += blockDim.x) a.out[(long long)blockIdx.x * a.B + j] = best[j];
}

// the last segment after each kept state: its optimal length
__global__ void k_beam_final(Table T, int n, const uint64_t *Kprev, int nb, uint64_t D, int *out) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b < nb) { const int d = find1(T, tcompose(Kprev[b], D, n)); out[b] = d < 0 ? 999 : d; }
}
