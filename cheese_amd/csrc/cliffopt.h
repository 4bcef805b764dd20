// Host side of `cliffopt JOB [--beam B]` (src/clifford.cu:285-385): the job file, the placements of every T gate
// (in the order of their tableaux, so the search is deterministic), the beam over them, the final choice and
// the optimal gate lists of the new segments.  Included by clifford.hip.

namespace {

struct CliffJob {
  int n = 0;
  std::vector<int> tq, td;                                   // T gates: qubit, dagger
  std::vector<std::vector<std::array<int, 3>>> seg;          // t + 1 segments of (kind, a, b)
};

// the job text (src/clifford.cu:224-238): "n t", t lines "q dagger", t + 1 lines "m gate q [q2] ..."
int read_cliff_job(const char *text, size_t len, CliffJob &J, std::string &err) {
  std::istringstream in(std::string(text, len));
  int t = -1;
  if (!(in >> J.n >> t) || J.n < 1 || J.n > 3 || t < 0 || t > 4096) { err = "bad job header"; return 2; }
  J.tq.resize(t);
  J.td.resize(t);
  for (int i = 0; i < t; i++)
    if (!(in >> J.tq[i] >> J.td[i]) || J.tq[i] < 0 || J.tq[i] >= J.n || (J.td[i] != 0 && J.td[i] != 1)) {
      err = "bad T gate line";
      return 2;
    }
  static const char *names[] = {"h", "s", "sdg", "x", "z", "cx", "y"};
  J.seg.resize(t + 1);
  for (auto &s : J.seg) {
    int m = -1;
    if (!(in >> m) || m < 0) { err = "bad segment length"; return 2; }
    for (int i = 0; i < m; i++) {
      std::string nm;
      if (!(in >> nm)) { err = "truncated segment"; return 2; }
      int k = -1;
      for (int j = 0; j < 7; j++) if (nm == names[j]) k = j;
      if (k < 0) { err = "unknown Clifford gate " + nm; return 2; }
      int a = 0, b = 0;
      if (!(in >> a) || a < 0 || a >= J.n) { err = "bad qubit"; return 2; }
      if (k == 5 && (!(in >> b) || b < 0 || b >= J.n || b == a)) { err = "bad cx target"; return 2; }
      s.push_back({k, a, b});
    }
  }
  return 0;
}

template <int NQ> int cliff_opt(chz_cliff *c, const CliffJob &J, int beam, double t0, char *out, size_t cap) {
  using chz_cl::Cand;
  using Num = chz_cl::Num<NQ>;
  const int n = NQ, t = (int)J.tq.size();
  std::vector<uint64_t> D(t + 1);                             // segment tableaux
  for (int j = 0; j <= t; j++) {
    uint64_t X = chz_cl::identity(n);
    for (const auto &g : J.seg[j]) X = chz_cl::apply(X, n, g[0], g[1], g[2]);
    D[j] = X;
  }
  std::vector<void *> owned;
  struct Guard { std::vector<void *> &o; ~Guard() { for (void *p : o) (void)cl_free(p); } } guard{owned};
  auto dalloc = [&](size_t bytes) -> void * {
    void *p = nullptr;
    if (cl_malloc(&p, std::max<size_t>(bytes, 8)) != hipSuccess) return nullptr;
    owned.push_back(p);
    return p;
  };
  // placements per qubit: the flagged signed Z images in order (candidate c is element zs[c / X_ALL] * X_ALL + c %
  // X_ALL), their places, and the placements' matrices
  struct Places { std::vector<uint32_t> zs; uint32_t *zpos = nullptr; chz_cl::PlaceMat *pm = nullptr; long long nm = 0; };
  std::vector<Places> places(n);
  constexpr int grid = 256;             // blocks of a beam step
  constexpr long long nbs = (Num::Z_ALL + CT_TILE - 1) / CT_TILE, nbu = (Num::Z_SYM + CT_TILE - 1) / CT_TILE;
  // the arrays whose sizes do not depend on the job, one block (an allocation each: 0.04 ms more for a 2-qubit job)
  size_t fixed = 0;
  auto part = [&](size_t bytes) { const size_t at = fixed; fixed += (bytes + 255) & ~(size_t)255; return at; };
  const size_t o_left = part(chz_cl::TOPK * 8), o_cost = part(chz_cl::TOPK * 4), o_hist = part(256 * 4),
               o_top = part((size_t)grid * chz_cl::TOPK * 8), o_bc = part((nbs + 1) * 8), o_bu = part((nbu + 1) * 8),
               o_tmp = part((nbs / SC_TILE + 8) * 8), o_zs = part((size_t)Num::Z_ALL * 4), o_zu = part((size_t)Num::Z_SYM * 4),
               o_zpos = part((size_t)Num::Z_ALL * 4 * n);
  uint8_t *const blk = (uint8_t *)dalloc(fixed);
  if (!blk) { chz_cl::g_err = "device memory"; return 5; }
  uint64_t *const d_left = (uint64_t *)(blk + o_left);
  int *const d_cost = (int *)(blk + o_cost);
  unsigned int *const d_hist = (unsigned int *)(blk + o_hist);
  unsigned long long *const d_top = (unsigned long long *)(blk + o_top);
  long long most = 0;                   // rows of a step per state
  {
    unsigned long long *const bc = (unsigned long long *)(blk + o_bc), *const bu = (unsigned long long *)(blk + o_bu);
    unsigned long long *const tmp = (unsigned long long *)(blk + o_tmp);
    uint32_t *const zs = (uint32_t *)(blk + o_zs), *const zu = (uint32_t *)(blk + o_zu);
    for (int q = 0; q < n; q++) {
      if (std::find(J.tq.begin(), J.tq.end(), q) == J.tq.end()) continue;
      Places &P = places[q];
      const chz_cl::FlagZs<NQ> fs{q};
      const chz_cl::FlagZ<NQ> fu{q};
      P.zpos = (uint32_t *)(blk + o_zpos) + (size_t)q * Num::Z_ALL;
      hipLaunchKernelGGL(k_flag_count<chz_cl::FlagZs<NQ>>, dim3((unsigned)nbs), dim3(CT_THREADS), 0, c->stream, fs,
                         (long long)Num::Z_ALL, bc);
      CLCHK(scan_excl(bc, nbs, tmp, c->stream));
      hipLaunchKernelGGL(k_scatter_idx<chz_cl::FlagZs<NQ>>, dim3((unsigned)nbs), dim3(CT_THREADS), 0, c->stream, fs,
                         (long long)Num::Z_ALL, bc, zs);
      hipLaunchKernelGGL(chz_cl::k_invert, dim3(64), dim3(256), 0, c->stream, zs, bc + nbs, P.zpos);
      hipLaunchKernelGGL(k_flag_count<chz_cl::FlagZ<NQ>>, dim3((unsigned)nbu), dim3(CT_THREADS), 0, c->stream, fu,
                         (long long)Num::Z_SYM, bu);
      CLCHK(scan_excl(bu, nbu, tmp, c->stream));
      hipLaunchKernelGGL(k_scatter_idx<chz_cl::FlagZ<NQ>>, dim3((unsigned)nbu), dim3(CT_THREADS), 0, c->stream, fu,
                         (long long)Num::Z_SYM, bu, zu);
      unsigned long long ns = 0, nu = 0;
      CLCHK(hipMemcpyAsync(&ns, bc + nbs, 8, hipMemcpyDeviceToHost, c->stream));
      CLCHK(hipMemcpyAsync(&nu, bu + nbu, 8, hipMemcpyDeviceToHost, c->stream));
      CLCHK(hipStreamSynchronize(c->stream));
      P.nm = (long long)nu * Num::X_SYM;
      P.zs.resize(ns);
      P.pm = (chz_cl::PlaceMat *)dalloc((size_t)P.nm * sizeof(chz_cl::PlaceMat));
      if (!P.pm) { chz_cl::g_err = "device memory"; return 5; }
      if (ns) CLCHK(hipMemcpyAsync(P.zs.data(), zs, ns * 4, hipMemcpyDeviceToHost, c->stream));
      if (P.nm)
        hipLaunchKernelGGL(chz_cl::k_place<NQ>, dim3((unsigned)std::min<long long>((P.nm + 255) / 256, 4096)), dim3(256), 0,
                           c->stream, zu, P.nm, q, P.pm);
      CLCHK(hipStreamSynchronize(c->stream));
      most = std::max(most, P.nm * 2);
    }
  }
  uint8_t *d_low = (uint8_t *)dalloc((size_t)most * beam);
  if (!d_low) { chz_cl::g_err = "device memory"; return 5; }
  // the beam over every T gate (src/clifford.cu:318-345)
  std::vector<std::vector<int>> parent(t), flips(t);
  std::vector<std::vector<Cand>> chosen(t);
  std::vector<uint64_t> hK(1, 0);
  std::vector<int> hcost(1, 0);
  for (int j = 0; j < t; j++) {
    const int q = J.tq[j], nb = (int)hK.size();
    const Places &P = places[q];
    const long long nc = (long long)P.zs.size() * Num::X_ALL, tot = nb * nc * 2;
    if (nc == 0) { chz_cl::g_err = "no placement for a T gate"; return 4; }
    std::vector<uint64_t> left(nb);
    for (int b = 0; b < nb; b++) left[b] = j == 0 ? D[0] : chz_cl::tcompose(hK[b], D[j], n);
    CLCHK(hipMemcpyAsync(d_left, left.data(), nb * 8, hipMemcpyHostToDevice, c->stream));
    CLCHK(hipMemcpyAsync(d_cost, hcost.data(), nb * 4, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(chz_cl::k_fill_u64, dim3(1), dim3(128), 0, c->stream, (unsigned long long *)d_hist, 128ll);
    chz_cl::BeamArgs ba{c->T, d_left, d_cost, nb, *std::min_element(hcost.begin(), hcost.end()), P.pm, P.nm, P.zpos, d_low,
                        d_hist, J.td[j], beam, d_top};
    const long long rows = nb * P.nm * 2;
    hipLaunchKernelGGL(chz_cl::k_beam_low<NQ>, dim3((unsigned)std::min<long long>((rows + 255) / 256, 4096)), dim3(256), 0,
                       c->stream, ba);
    const int blocks = (int)std::min<long long>(grid, (rows + 15) / 16);
    hipLaunchKernelGGL(chz_cl::k_beam<NQ>, dim3(blocks), dim3(256), 0, c->stream, ba);
    CLCHK(hipGetLastError());
    std::vector<unsigned long long> top((size_t)blocks * beam);
    CLCHK(hipMemcpyAsync(top.data(), d_top, top.size() * 8, hipMemcpyDeviceToHost, c->stream));
    CLCHK(hipStreamSynchronize(c->stream));
    const int keep = (int)std::min<long long>(beam, tot);
    std::partial_sort(top.begin(), top.begin() + keep, top.end());
    parent[j].resize(keep);
    flips[j].resize(keep);
    chosen[j].resize(keep);
    std::vector<uint64_t> nk(keep);
    std::vector<int> ncost(keep);
    for (int i = 0; i < keep; i++) {
      const int b = (int)((top[i] >> 32) & 0xff);
      const long long c2 = (long long)(top[i] & 0xffffffffull);
      const uint64_t cand = (uint64_t)(c2 >> 1);
      chosen[j][i] = chz_cl::make_cand(Num::element((uint64_t)P.zs[cand / Num::X_ALL] * Num::X_ALL + cand % Num::X_ALL), n, q);
      parent[j][i] = b;
      flips[j][i] = (int)(c2 & 1);
      ncost[i] = (int)(top[i] >> 40);
    }
    for (int i = 0; i < keep; i++) nk[i] = chosen[j][i].K;
    hK = nk;
    hcost = ncost;
  }
  // the final segment after each kept state; the best total, first in state order
  int best = 0, bestv = 1 << 30;
  if (t > 0) {
    int *const d_fin = d_cost;          // (the last step has read its costs)
    CLCHK(hipMemcpyAsync(d_left, hK.data(), hK.size() * 8, hipMemcpyHostToDevice, c->stream));
    hipLaunchKernelGGL(chz_cl::k_beam_final, dim3(((int)hK.size() + 63) / 64), dim3(64), 0, c->stream, c->T, n, d_left,
                       (int)hK.size(), D[t], d_fin);
    std::vector<int> fin(hK.size());
    CLCHK(hipMemcpyAsync(fin.data(), d_fin, fin.size() * 4, hipMemcpyDeviceToHost, c->stream));
    CLCHK(hipStreamSynchronize(c->stream));
    for (size_t b = 0; b < hK.size(); b++)
      if (hcost[b] + fin[b] < bestv) { bestv = hcost[b] + fin[b]; best = (int)b; }
  }
  std::vector<Cand> K(t);
  std::vector<int> flip(t), dag(t);
  for (int j = t - 1, b = best; j >= 0; j--) { K[j] = chosen[j][b]; flip[j] = flips[j][b]; b = parent[j][b]; }
  for (int j = 0; j < t; j++) {          // the T actually placed: its dagger after the sign and the flip
    const int d0 = J.td[j] ^ K[j].neg;
    if (flip[j]) K[j].Kinv = chz_cl::flipped_inv(K[j], d0, n);
    dag[j] = d0 ^ flip[j];
  }
  // the new segments K_{j-1} then D_j then K_j^-1, each read back as an optimal gate list
  std::vector<uint64_t> X(t + 1);
  for (int j = 0; j <= t; j++) {
    uint64_t x = j > 0 ? chz_cl::tcompose(K[j - 1].K, D[j], n) : D[j];
    if (j < t) x = chz_cl::tcompose(x, K[j].Kinv, n);
    X[j] = x;
  }
  constexpr int MAXW = 32;
  std::vector<uint8_t> words((size_t)(t + 1) * MAXW);
  std::vector<int> lens(t + 1);
  if (const int rc = chz_cliff_readback(c, X.data(), t + 1, MAXW, words.data(), lens.data())) return rc;
  int total = 0, orig = 0;
  for (int j = 0; j <= t; j++) {
    if (lens[j] < 0) { chz_cl::g_err = "segment not in the table"; return 4; }
    total += lens[j];
    orig += (int)J.seg[j].size();
  }
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count() - t0;
  char buf[160];
  std::snprintf(buf, sizeof buf, "{\"clifford_gates\": %d, \"clifford_gates_before\": %d, \"t_gates\": %d, \"seconds\": %.2f}\n",
                total, orig, t, secs);
  std::string s = buf;
  static const char *gn[] = {"h", "s", "sdg", "x", "z", "cx", "y"};
  for (int j = 0; j <= t; j++) {
    for (int i = 0; i < lens[j]; i++) {
      const int g = words[(size_t)j * MAXW + i];
      if (c->G.k[g] == 5) std::snprintf(buf, sizeof buf, "cx %d %d\n", c->G.a[g], c->G.b[g]);
      else std::snprintf(buf, sizeof buf, "%s %d\n", gn[c->G.k[g]], c->G.a[g]);
      s += buf;
    }
    if (j < t) {
      std::snprintf(buf, sizeof buf, "%s %d\n", dag[j] ? "tdg" : "t", K[j].qp);
      s += buf;
    }
  }
  if (!out || s.size() + 1 > cap) { chz_cl::g_err = "output buffer too small (" + std::to_string(s.size() + 1) + " bytes)"; return 4; }
  s.copy(out, s.size());
  out[s.size()] = 0;
  return 0;
}

}  // namespace

extern "C" int chz_cliff_opt(chz_cliff *c, const char *job, size_t len, int beam, char *out, size_t cap) {
  chz::RelaxedCapture relaxed;
  const double t0 = std::chrono::duration<double>(std::chrono::steady_clock::now().time_since_epoch()).count();
  CliffJob J;
  std::string err;
  if (const int rc = read_cliff_job(job, len, J, err)) { chz_cl::g_err = err; return rc; }
  if (J.n != c->n) { chz_cl::g_err = "the job's qubit count differs from the table's"; return 3; }
  beam = std::max(1, std::min(chz_cl::TOPK - 1, beam));
  CLCHK(hipSetDevice(c->device));
  return J.n == 1 ? cliff_opt<1>(c, J, beam, t0, out, cap) : J.n == 2 ? cliff_opt<2>(c, J, beam, t0, out, cap)
                                                                      : cliff_opt<3>(c, J, beam, t0, out, cap);
}
