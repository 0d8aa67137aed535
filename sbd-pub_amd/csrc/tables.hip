// Excitation tables, the diagonal and the basis sign.
//
// Table construction follows the semantics of GenerateExcitation
// (chemistry/tpb/helper.h:185-323): for every bra string, every ket string of
// the same set at Hamming distance 2 (single) or 4 (double), in ascending ket
// index.  One 64-lane wavefront owns one bra string and sweeps the kets 64 at
// a time; popcount of the XOR gives the distance and the wave ballot + a
// masked popcount give each match its slot, so the order is ascending
// without sorting.
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <exception>
#include <memory>
#include <mutex>

#include "common.h"

// host code only: the population count as an instruction
#ifdef __HIP_DEVICE_COMPILE__
#define SBDX_POPCNT
#else
#define SBDX_POPCNT __attribute__((target("popcnt")))
#endif

namespace sbdx {

// fn(i) for i in [0, n) on up to 16 host threads (work independent per i);
// an exception of any of them is rethrown here once all have ended.  The call
// ends with the last item, not with the last thread: a thread that the
// system starts late, on a busy host a scheduler's tick of 3 ms later, finds
// nothing left, and the context joins it afterwards (waiting for it here, the
// first product of 300 x 289 strings took 3.8 ms beside a BLAS library's
// spinning threads, 0.6 this way).  Such a thread touches the shared counters
// alone; fn lives as long as any item is worked on.
template <typename F>
static void parallel_for(Context &c, int n, const F &fn) {
  struct Shared {
    std::atomic<int> next{0};
    std::mutex mu;
    std::condition_variable ended;
    int done = 0;
    std::exception_ptr err;
  };
  if (n <= 0) return;
  auto sh = std::make_shared<Shared>();
  auto worker = [sh, n, f = &fn]() {
    for (int i = sh->next++; i < n; i = sh->next++) {
      std::exception_ptr e;
      try {
        (*f)(i);
      } catch (...) {
        e = std::current_exception();
      }
      std::lock_guard<std::mutex> lock(sh->mu);
      if (e && !sh->err) {
        sh->err = e;
        const int first = sh->next.exchange(n);  // nobody takes the rest
        if (first < n) sh->done += n - first;
      }
      if (++sh->done == n) sh->ended.notify_all();
    }
  };
  if (c.helpers.t.size() >= 32) c.helpers.join();
  const int nthr = std::max(1, std::min({16, (int)std::thread::hardware_concurrency(), n}));
  try {
    for (int i = 1; i < nthr; i++) c.helpers.t.emplace_back(worker);
  } catch (...) {  // no more threads: those that run and this one do the work
  }
  worker();
  std::unique_lock<std::mutex> lock(sh->mu);
  sh->ended.wait(lock, [&]() { return sh->done == n; });
  if (sh->err) std::rethrow_exception(sh->err);
}

__device__ __forceinline__ double parity1(uint64_t s, int a, int b) {
  // Reference parity rule (chemistry/basic/determinants.h:230-281) on one
  // string: bits in [lo, hi), one more flip when bit lo is set.
  int lo = a < b ? a : b, hi = a < b ? b : a;
  uint64_t mask = ((1ull << hi) - 1ull) ^ ((1ull << lo) - 1ull);
  int n = __popcll(s & mask) + (int)((s >> lo) & 1ull);
  return (n & 1) ? -1.0 : 1.0;
}

__global__ void __launch_bounds__(256) k_table_count(const uint64_t *__restrict__ s, int n,
                                                     uint32_t *__restrict__ cs,
                                                     uint32_t *__restrict__ cd) {
  const int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  if (wave >= n) return;  // uniform per wave
  const uint64_t me = s[wave];
  uint32_t a = 0, b = 0;
  for (int j0 = 0; j0 < n; j0 += 64) {
    const int j = j0 + lane;
    const int d = (j < n) ? __popcll(me ^ s[j]) : 0;
    a += (uint32_t)__popcll(__ballot(d == 2));
    b += (uint32_t)__popcll(__ballot(d == 4));
  }
  if (lane == 0) {
    cs[wave] = a;
    cd[wave] = b;
  }
}

__global__ void __launch_bounds__(256) k_table_fill(
    const uint64_t *__restrict__ s, int n, int L, const uint64_t *__restrict__ s_off,
    const uint64_t *__restrict__ d_off, const double *__restrict__ eri,
    const double *__restrict__ h1, uint64_t *__restrict__ s_ent, double *__restrict__ s_val,
    uint32_t *__restrict__ d_ket, uint32_t *__restrict__ d_orb, double *__restrict__ d_val) {
  const int wave = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int lane = threadIdx.x & 63;
  if (wave >= n) return;
  const int K = L * L;
  const uint64_t me = s[wave];
  const uint64_t below = (1ull << lane) - 1ull;
  uint64_t ps = s_off[wave], pd = d_off[wave];
  for (int j0 = 0; j0 < n; j0 += 64) {
    const int j = j0 + lane;
    const uint64_t sj = (j < n) ? s[j] : me;
    const int d = __popcll(me ^ sj);
    const uint64_t m2 = __ballot(d == 2), m4 = __ballot(d == 4);
    if (d == 2) {
      const uint64_t pos = ps + (uint64_t)__popcll(m2 & below);
      const int p = __ffsll((unsigned long long)(me & ~sj)) - 1;
      const int q = __ffsll((unsigned long long)(sj & ~me)) - 1;
      const double sg = parity1(me, p, q);
      const int pq = p * L + q;
      double F = h1[pq];
      uint64_t occ = me;
      while (occ) {
        const int k = __ffsll((unsigned long long)occ) - 1;
        occ &= occ - 1;
        F += eri[(size_t)pq * K + k * L + k] - eri[(size_t)(p * L + k) * K + k * L + q];
      }
      s_ent[pos] = (uint64_t)j | ((uint64_t)pq << 32) | (sg < 0 ? (1ull << 63) : 0ull);
      s_val[pos] = sg * F;
    } else if (d == 4) {
      const uint64_t pos = pd + (uint64_t)__popcll(m4 & below);
      const uint64_t cr = me & ~sj, an = sj & ~me;
      const int i = __ffsll((unsigned long long)cr) - 1, jj = 63 - __clzll(cr);
      const int a = __ffsll((unsigned long long)an) - 1, b = 63 - __clzll(an);
      double sg = parity1(me, i, a) * parity1(me, jj, b);
      if (a > jj || b < i) sg = -sg;
      const double v = eri[(size_t)(a * L + i) * K + b * L + jj] -
                       eri[(size_t)(a * L + jj) * K + b * L + i];
      d_ket[pos] = (uint32_t)j;
      d_orb[pos] = (uint32_t)i | ((uint32_t)jj << 8) | ((uint32_t)a << 16) | ((uint32_t)b << 24);
      d_val[pos] = sg * v;
    }
    ps += (uint64_t)__popcll(m2);
    pd += (uint64_t)__popcll(m4);
  }
}

// Per-string pieces of the diagonal: e1[x] = sum_p h_pp + sum_{p<q}
// ((pp|qq) - (pq|qp)) and jsum[x][r] = sum_{p in x} (pp|rr).
__global__ void __launch_bounds__(256) k_string_energy(const uint64_t *__restrict__ s, int n,
                                                       int L, const double *__restrict__ eri,
                                                       const double *__restrict__ h1,
                                                       double *__restrict__ e1,
                                                       double *__restrict__ jsum) {
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= n) return;
  const int K = L * L;
  const uint64_t str = s[x];
  double e = 0.0;
  for (int p = 0; p < L; p++) {
    if (!((str >> p) & 1ull)) continue;
    e += h1[p * L + p];
    for (int q = p + 1; q < L; q++) {
      if (!((str >> q) & 1ull)) continue;
      e += eri[(size_t)(p * L + p) * K + q * L + q] - eri[(size_t)(p * L + q) * K + q * L + p];
    }
  }
  e1[x] = e;
  for (int r = 0; r < L; r++) {
    double j = 0.0;
    for (int p = 0; p < L; p++)
      if ((str >> p) & 1ull) j += eri[(size_t)(p * L + p) * K + r * L + r];
    jsum[(size_t)x * L + r] = j;
  }
}

// hii[ia*nb+ib] = I0 + e1a[ia] + e1b[ib] + sum_{r in beta(ib)} jsum_a[ia][r]
// (ZeroExcite, chemistry/basic/determinants.h:434-457, split by spin).
// canon != 0 (equal string sets, shared tables): element (ia, ib) with
// ib < ia is evaluated as (ib, ia), so hii is bitwise symmetric and the
// spin-flip sectors (x = +-x^T) stay exact under hii * x.
__global__ void __launch_bounds__(256) k_diag(int nb, int nchunk, int L, double I0, int canon,
                                              const uint64_t *__restrict__ bstr,
                                              const double *__restrict__ e1a,
                                              const double *__restrict__ e1b,
                                              const double *__restrict__ jsa,
                                              double *__restrict__ hii) {
  const int ia = blockIdx.x / nchunk;
  const int ib = (blockIdx.x % nchunk) * blockDim.x + threadIdx.x;
  if (ib >= nb) return;
  const bool swap = canon && ib < ia;
  const double *j = jsa + (size_t)(swap ? ib : ia) * L;
  uint64_t occ = bstr[swap ? ia : ib];
  double acc = 0.0;
  while (occ) {
    const int r = __ffsll((unsigned long long)occ) - 1;
    occ &= occ - 1;
    acc += j[r];
  }
  hii[(size_t)ia * nb + ib] = I0 + (e1a[ia] + e1b[ib]) + acc;
}

// out = S * in, S(ia,ib) = (-1)^#{(p in alpha, r in beta): r < p}: the sign
// between the interleaved (reference) and the alpha-first basis.
template <bool ACC>
__global__ void __launch_bounds__(256) k_sign(int nb, int nchunk, const uint64_t *__restrict__ astr,
                                              const uint64_t *__restrict__ bstr,
                                              const double *__restrict__ in,
                                              double *__restrict__ out) {
  const int ia = blockIdx.x / nchunk;
  const int ib = (blockIdx.x % nchunk) * blockDim.x + threadIdx.x;
  if (ib >= nb) return;
  uint64_t a = astr[ia];
  const uint64_t b = bstr[ib];
  int cnt = 0;
  while (a) {
    const int p = __ffsll((unsigned long long)a) - 1;
    a &= a - 1;
    cnt += __popcll(b & ((1ull << p) - 1ull));
  }
  const size_t idx = (size_t)ia * nb + ib;
  const double v = (cnt & 1) ? -in[idx] : in[idx];
  out[idx] = ACC ? out[idx] + v : v;
}

static inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

void build_spin_tables(Context &c, SpinTables &t, const std::vector<uint64_t> &strs) {
  const int n = (int)strs.size();
  t.n = n;
  t.str = (uint64_t *)dalloc(c, sizeof(uint64_t) * n);
  SBDX_HIP(hipMemcpyAsync(t.str, strs.data(), sizeof(uint64_t) * n, hipMemcpyHostToDevice, c.stream));
  uint32_t *cnt = (uint32_t *)dalloc(c, sizeof(uint32_t) * 2 * (size_t)n);
  {
    ProfScope ps(c, "table_count");
    hipLaunchKernelGGL(k_table_count, dim3(cdiv((size_t)n * 64, 256)), dim3(256), 0, c.stream,
                       t.str, n, cnt, cnt + n);
    check_launch("k_table_count");
  }
  std::vector<uint32_t> hc(2 * (size_t)n);
  SBDX_HIP(hipMemcpyAsync(hc.data(), cnt, sizeof(uint32_t) * 2 * n, hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipStreamSynchronize(c.stream));
  std::vector<uint64_t> so(n + 1, 0), dof(n + 1, 0);
  size_t mx = 0;
  for (int i = 0; i < n; i++) {
    so[i + 1] = so[i] + hc[i];
    dof[i + 1] = dof[i] + hc[n + i];
    if (hc[i] > mx) mx = hc[i];
  }
  t.ns = so[n];
  t.nd = dof[n];
  t.max_s = mx;
  t.s_off = (uint64_t *)dalloc(c, sizeof(uint64_t) * (n + 1));
  t.d_off = (uint64_t *)dalloc(c, sizeof(uint64_t) * (n + 1));
  SBDX_HIP(hipMemcpyAsync(t.s_off, so.data(), sizeof(uint64_t) * (n + 1), hipMemcpyHostToDevice, c.stream));
  SBDX_HIP(hipMemcpyAsync(t.d_off, dof.data(), sizeof(uint64_t) * (n + 1), hipMemcpyHostToDevice, c.stream));
  t.s_ent = (uint64_t *)dalloc(c, sizeof(uint64_t) * (t.ns + 1));
  t.s_val = (double *)dalloc(c, sizeof(double) * (t.ns + 1));
  t.d_ket = (uint32_t *)dalloc(c, sizeof(uint32_t) * (t.nd + 1));
  t.d_orb = (uint32_t *)dalloc(c, sizeof(uint32_t) * (t.nd + 1));
  t.d_val = (double *)dalloc(c, sizeof(double) * (t.nd + 1));
  {
    ProfScope ps(c, "table_fill");
    hipLaunchKernelGGL(k_table_fill, dim3(cdiv((size_t)n * 64, 256)), dim3(256), 0, c.stream, t.str,
                       n, c.L, t.s_off, t.d_off, c.eri, c.h1, t.s_ent, t.s_val, t.d_ket, t.d_orb,
                       t.d_val);
    check_launch("k_table_fill");
  }
  t.e1 = (double *)dalloc(c, sizeof(double) * n);
  t.jsum = (double *)dalloc(c, sizeof(double) * (size_t)n * c.L);
  hipLaunchKernelGGL(k_string_energy, dim3(cdiv(n, 256)), dim3(256), 0, c.stream, t.str, n, c.L,
                     c.eri, c.h1, t.e1, t.jsum);
  check_launch("k_string_energy");
}

// Sliced-ELL copy of the singles (see SpinTables::ell).  Needs kets < 2^16
// and pq < 2^15; otherwise has_ell stays false and the CSR kernels run.
// Order of one 64-row slice's entries (position k of lane l at
// out[64*k + l]).  The mixed kernels read x[.., ket] and V[.., pq] from LDS
// at the indices of entry k of all 64 lanes at once, and the row sums do
// not depend on the entry order, so entries are dealt greedily: at each k,
// lane by lane, the remaining entry whose ket and pq residues are least
// used so far at this k.  Measured gfx950 LDS bank rule: 4- and 8-byte
// reads are served 32 lanes at a time and two distinct addresses of one
// half-wavefront conflict when their element indices agree mod 32; 16-byte
// reads (4 FP32 or 2 FP64 pairs per entry) are served 16 lanes at a time and
// conflict when the indices agree mod 16 within the quarter-wavefront.  The
// cost of a candidate is 2 x (uses of its residues mod 16 in the lane's
// quarter) + (uses of its residues mod 32 in the lane's half), which keeps
// both rules nearly balanced.  Padding entries (pq = pad, a zero in every
// staged ERI row, one shared address) take an unused ket residue below nb.
static void schedule_slice(std::vector<uint32_t> *rows, uint32_t len, uint32_t pad_pq, uint32_t nb,
                           uint32_t *out) {
  for (uint32_t k = 0; k < len; k++) {
    uint8_t hj[32], hv[32], qj[16], qv[16];
    for (int l = 0; l < 64; l++) {
      if ((l & 31) == 0) {
        std::fill(hj, hj + 32, 0);
        std::fill(hv, hv + 32, 0);
      }
      if ((l & 15) == 0) {
        std::fill(qj, qj + 16, 0);
        std::fill(qv, qv + 16, 0);
      }
      std::vector<uint32_t> &R = rows[l];
      uint32_t w;
      if (R.empty()) {
        int best = 0, bc = 1 << 30;
        for (int j = 0; j < 32; j++) {
          const int cost = 2 * qj[j & 15] + hj[j];
          if (cost < bc) {
            bc = cost;
            best = j;
          }
        }
        const uint32_t jb = nb > 32 ? (uint32_t)best : (uint32_t)best % nb;
        w = jb | (pad_pq << 16);
      } else {
        size_t bi = 0;
        int bc = 1 << 30;
        for (size_t i = 0; i < R.size(); i++) {
          const uint32_t e = R[i], v = e >> 16;
          const int cost = 2 * (qj[e & 15] + qv[v & 15]) + hj[e & 31] + hv[v & 31];
          if (cost < bc) {
            bc = cost;
            bi = i;
            if (cost == 0) break;
          }
        }
        w = R[bi];
        R[bi] = R.back();
        R.pop_back();
        qv[(w >> 16) & 15]++;
        hv[(w >> 16) & 31]++;
      }
      qj[w & 15]++;
      hj[w & 31]++;
      out[(size_t)64 * k + l] = w;
    }
  }
}

// Slices of the sliced-ELL layout with the rows of t taken in `order` (64
// rows per slice); results in host vectors, returns the number of entries.
static uint64_t ell_slices(const SpinTables &t, const std::vector<uint64_t> &off,
                           const std::vector<uint32_t> &order, std::vector<uint32_t> &perm,
                           std::vector<uint32_t> &sl_len, std::vector<uint64_t> &sl_off) {
  const int n = t.n;
  const int nsl = (n + 63) / 64;
  perm.assign((size_t)nsl * 64, 0xffffffffu);
  sl_len.assign(nsl, 0);
  sl_off.assign(nsl, 0);
  uint64_t total = 0;
  for (int s = 0; s < nsl; s++) {
    uint32_t mx = 0;
    for (int l = 0; l < 64 && s * 64 + l < n; l++) {
      const uint32_t r = order[s * 64 + l];
      perm[(size_t)s * 64 + l] = r;
      mx = std::max<uint32_t>(mx, (uint32_t)(off[r + 1] - off[r]));
    }
    sl_len[s] = mx;
    sl_off[s] = total;
    total += (uint64_t)mx * 64;
  }
  return total;
}

// Packed entries of the staged mixed kernel (SpinTables::ell2): bits 4..18
// hold K + ket, the LDS element of the ket's staged value (the staged ERI
// row occupies elements 0..K-1, the ket row K..K+nb-1, a zero at K+nb),
// so (w & 0x7fff0) is its byte offset for 16-byte elements; bits 19..30
// hold pq, (w >> 15) & 0xfff0 its byte offset; bit 31 the sign.  Padding
// entries read the zero ket element and ERI element 0, one address shared
// by every padding lane (an LDS broadcast).
//
// Dealing a slice's entries to positions.  Measured on gfx950 with the
// SQ_LDS_BANK_CONFLICT counter over per-lane index patterns (lanes in the
// same coset of a 2-dimensional subspace of lane-index bits sharing a
// residue, for every pair of bits): a 16-byte LDS read of a wavefront takes
// 4 cycles when conflict-free, lane l being served in lane group
// 2 * bit5(l) + (bit4 ^ bit3 ^ bit2)(l) (16 lanes per group), and two
// distinct addresses of one group conflict when their 16-byte element
// indices agree mod 16 (64 banks of 4 bytes); the cycles of one read are the
// sum over the 4 groups of the largest number of distinct addresses sharing
// a residue.  The groups are
// independent: for each, every position takes one entry per lane (or, for a
// lane with fewer entries than positions left, the shared padding address),
// and a depth-first search (the lane with the fewest options first, entries
// with the most heavily loaded residues first, a node budget) looks for a
// position whose ket residues and ERI residues each repeat at most (cx, cw)
// times in the group, trying (1,1), then (1,2) and (2,1), and so on; an
// unbounded greedy choice ends it.  On the norb-36 workload this takes the
// modelled cost of one read from 8.9 cycles (dealing that ignores the lane
// grouping) to 5.2 (4 without conflicts).  4- and 8-byte reads follow
// another rule (schedule_slice_packed), dealt by the same search.
namespace qsched {
// NL lanes per group, NR residues (16 or 32; NL == NR here)
template <int NR>
struct Lane {
  static constexpr int W = NR * NR / 64;
  std::vector<uint32_t> ent;
  uint16_t cnt[NR * NR];  // entries per (x, w) residue pair
  uint64_t have[W];       // bit x NR + w: some entry has residues (x, w)
};
template <int NR>
static inline int rx(uint32_t w) { return (w >> 4) & (NR - 1); }
template <int NR>
static inline int rw(uint32_t w) { return (w >> 19) & (NR - 1); }
template <int NL, int NR>
struct Search {
  static constexpr int W = NR * NR / 64, XW = 64 / NR;  // residues x per word of a pair set
  Lane<NR> *L;
  int remx[NR], remw[NR];
  uint8_t ux[NR], uw[NR];
  int cx, cw;
  int padx, padw;
  bool padused;
  long nodes, limit;
  int pick[NL];  // pair index x*NR+w, or -1 idle
  bool need[NL], done[NL];
  bool fits(int x, int w) const { return ux[x] < cx && uw[w] < cw; }
  SBDX_POPCNT bool dfs(int depth) {
    if (depth == NL) return true;
    if (++nodes > limit) return false;
    // the pairs whose residues are both below their bounds
    uint64_t open[W], wf = 0;
    for (int w = 0; w < NR; w++)
      if (uw[w] < cw) wf |= 1ull << w;
    for (int i = 0; i < W; i++) {
      open[i] = 0;
      for (int q = 0; q < XW; q++)
        if (ux[i * XW + q] < cx) open[i] |= wf << (q * NR);
    }
    int bl = -1, bn = 1 << 30;
    for (int l = 0; l < NL; l++) {
      if (done[l]) continue;
      int n = need[l] ? 0 : 1;
      for (int i = 0; i < W; i++) n += __builtin_popcountll(L[l].have[i] & open[i]);
      if (n < bn) { bn = n; bl = l; }
    }
    if (bn == 0) return false;
    const int l = bl;
    done[l] = true;
    // its candidates, the most loaded residues first (then the lowest pair);
    // most searches take the first, so the order is found as it is needed
    uint32_t cand[NR * NR];
    int nc = 0;
    for (int i = 0; i < W; i++)
      for (uint64_t m = L[l].have[i] & open[i]; m; m &= m - 1) {
        const int p = 64 * i + __builtin_ctzll(m);
        cand[nc++] = ((uint32_t)(remx[p / NR] + remw[p % NR]) << 10) | (uint32_t)(NR * NR - 1 - p);
      }
    for (int i = 0; i < nc; i++) {
      int best = i;
      for (int j = i + 1; j < nc; j++)
        if (cand[j] > cand[best]) best = j;
      std::swap(cand[i], cand[best]);
      const int p = NR * NR - 1 - (int)(cand[i] & (NR * NR - 1)), x = p / NR, w = p % NR;
      ux[x]++; uw[w]++;
      pick[l] = p;
      if (dfs(depth + 1)) return true;
      ux[x]--; uw[w]--;
      if (nodes > limit) break;
    }
    if (!need[l]) {
      const bool was = padused;
      if (was || fits(padx, padw)) {
        if (!was) { ux[padx]++; uw[padw]++; padused = true; }
        pick[l] = -1;
        if (dfs(depth + 1)) return true;
        if (!was) { ux[padx]--; uw[padw]--; padused = false; }
      }
    }
    done[l] = false;
    return false;
  }
};
// rows(lane, v): puts lane's entries into v.  Entry k of lane l goes to
// out[256 (k / 4) + 4 l + k % 4]: groups of 4 positions, each lane-major.
template <int NL, int NR, typename F>
static void deal_group(const F &rows, const int *lanes, uint32_t len, uint32_t pad, uint32_t *out, long limit) {
  static_assert(NR * NR <= 1024, "a pair index takes 10 bits");
  std::vector<Lane<NR>> L(NL);
  Search<NL, NR> s;
  s.L = L.data();
  std::fill(s.remx, s.remx + NR, 0);
  std::fill(s.remw, s.remw + NR, 0);
  for (int l = 0; l < NL; l++) {
    rows(lanes[l], L[l].ent);
    std::fill(L[l].cnt, L[l].cnt + NR * NR, 0);
    std::fill(L[l].have, L[l].have + Lane<NR>::W, 0ull);
    for (uint32_t w : L[l].ent) {
      const int p = rx<NR>(w) * NR + rw<NR>(w);
      L[l].cnt[p]++;
      L[l].have[p / 64] |= 1ull << (p % 64);
      s.remx[p / NR]++;
      s.remw[p % NR]++;
    }
  }
  s.padx = rx<NR>(pad);
  s.padw = rw<NR>(pad);
  static const int caps[][2] = {{1, 1}, {1, 2}, {2, 1}, {2, 2}, {2, 3}, {3, 2}, {3, 3}};
  const int ncaps = sizeof(caps) / sizeof(caps[0]);
  for (uint32_t k = 0; k < len; k++) {
    const uint32_t left = len - k;
    for (int l = 0; l < NL; l++) s.need[l] = L[l].ent.size() >= left;
    bool ok = false;
    for (int c = 0; c < ncaps && !ok; c++) {
      s.cx = caps[c][0];
      s.cw = caps[c][1];
      std::fill(s.ux, s.ux + NR, 0);
      std::fill(s.uw, s.uw + NR, 0);
      std::fill(s.done, s.done + NL, false);
      s.padused = false;
      s.nodes = 0;
      s.limit = limit;
      ok = s.dfs(0);
    }
    if (!ok) {
      // unbounded: lane by lane, the pair minimizing the larger use count
      std::fill(s.ux, s.ux + NR, 0);
      std::fill(s.uw, s.uw + NR, 0);
      bool pu = false;
      for (int l = 0; l < NL; l++) {
        if (L[l].ent.empty()) {
          s.pick[l] = -1;
          if (!pu) { s.ux[s.padx]++; s.uw[s.padw]++; pu = true; }
          continue;
        }
        long best = 1L << 60;
        int bp = 0;
        for (int p = 0; p < NR * NR; p++) {
          if (!L[l].cnt[p]) continue;
          const int x = p / NR, w = p % NR;
          const long sc = (long)std::max(s.ux[x], s.uw[w]) * 1000000 + (long)(s.ux[x] + s.uw[w]) * 1000 -
                          (s.remx[x] + s.remw[w]);
          if (sc < best) { best = sc; bp = p; }
        }
        s.pick[l] = bp;
        s.ux[bp / NR]++;
        s.uw[bp % NR]++;
      }
    }
    for (int l = 0; l < NL; l++) {
      uint32_t w = pad;
      if (s.pick[l] >= 0 && !L[l].ent.empty()) {
        const int p = s.pick[l];
        auto &E = L[l].ent;
        for (size_t i = 0; i < E.size(); i++)
          if (rx<NR>(E[i]) * NR + rw<NR>(E[i]) == p) { w = E[i]; E[i] = E.back(); E.pop_back(); break; }
        if (--L[l].cnt[p] == 0) L[l].have[p / 64] &= ~(1ull << (p % 64));
        s.remx[p / NR]--;
        s.remw[p % NR]--;
      }
      out[256 * (size_t)(k / 4) + 4 * lanes[l] + k % 4] = w;
    }
  }
}
}  // namespace qsched

// The packed entries of lane group g of one slice (rows(lane, v): a lane's
// entries): for 16-byte reads one of the 4 measured lane groups of 16 lanes
// with residues mod 16; for 4- and 8-byte reads one of the two half-waves
// with residues mod 32 (measured with the same probe: lanes of different
// half-waves never conflict, and two distinct addresses of one half-wave
// conflict when their element indices agree mod 32).
static int lane_groups(bool wide) { return wide ? 4 : 2; }
template <typename F>
static void schedule_slice_packed(const F &rows, int g, uint32_t len, uint32_t pad, uint32_t *out, bool wide) {
  if (wide) {
    int lanes[16], n = 0;
    for (int l = 0; l < 64; l++)
      if (((l >> 5) & 1) * 2 + (((l >> 4) ^ (l >> 3) ^ (l >> 2)) & 1) == g) lanes[n++] = l;
    qsched::deal_group<16, 16>(rows, lanes, len, pad, out, 200);
  } else {
    int lanes[32];
    for (int l = 0; l < 32; l++) lanes[l] = 32 * g + l;
    qsched::deal_group<32, 32>(rows, lanes, len, pad, out, 200);
  }
}

static void download_singles(Context &c, const SpinTables &t, std::vector<uint64_t> &off,
                             std::vector<uint64_t> &ent) {
  off.resize(t.n + 1);
  ent.resize(t.ns);
  SBDX_HIP(hipMemcpyAsync(off.data(), t.s_off, sizeof(uint64_t) * (t.n + 1), hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipMemcpyAsync(ent.data(), t.s_ent, sizeof(uint64_t) * t.ns, hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipStreamSynchronize(c.stream));
}

void build_singles_ell(Context &c, SpinTables &t) {
  t.has_ell = false;
  if (t.n > 65536 || c.K >= 32768) return;
  const int n = t.n;
  std::vector<uint64_t> off, ent;
  download_singles(c, t, off, ent);
  std::vector<uint32_t> order(n);
  for (int i = 0; i < n; i++) order[i] = (uint32_t)i;
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    return (off[a + 1] - off[a]) > (off[b + 1] - off[b]);
  });
  std::vector<uint32_t> perm, sl_len;
  std::vector<uint64_t> sl_off;
  const uint64_t total = ell_slices(t, off, order, perm, sl_len, sl_off);
  const int nsl = (int)sl_len.size();
  // 4 x 64 padding entries past the end: the mixed kernel prefetches the
  // next 4 positions of a slice unconditionally (past a slice's end it
  // reads the next slice's entries or these, and never uses them)
  std::vector<uint32_t> ell(total + 4 * 64 + 1, (uint32_t)c.K << 16);
  // the packed form for k_mixed_ell (same rows, slices and lengths)
  t.has_ell2 = false;
  t.has_ell3 = false;
  const bool packed = c.K <= 4096 && (size_t)c.K + (size_t)n <= 32767;
  const uint32_t pad2 = ((uint32_t)(c.K + n)) << 4;
  // the reads the kernel will make: 16-byte values when four FP32 pairs fit
  // in LDS (the autotuner's choice whenever they do), else 4- or 8-byte ones
  const bool wide = (size_t)4 * ((size_t)c.K + n + 1) * sizeof(float) <= c.lds_limit;
  // groups of 4 positions: slice lengths rounded up to a multiple of 4, each
  // group stored lane-major (lane l's 4 words contiguous, one 16-byte load),
  // plus 2 groups of padding past the end for the kernel's prefetch
  std::vector<uint32_t> sl_len2(nsl);
  std::vector<uint64_t> sl_off2(nsl);
  uint64_t total2 = 0;
  for (int sl = 0; sl < nsl; sl++) {
    sl_len2[sl] = (sl_len[sl] + 3) & ~3u;
    sl_off2[sl] = total2;
    total2 += (uint64_t)sl_len2[sl] * 64;
  }
  // the signed-triangle form: dealt in the ell2 word layout with the ket
  // element at 2048 + ket (the kernel's ket rows start at byte 32768 = 2048
  // 16-byte elements, so residues match the LDS addresses) and the signed
  // triangle index in the pq field, then repacked
  const bool triangle = packed && c.eri_rs_sym && c.Kt <= 1024 && n < 8192 && wide;
  const uint32_t pad3 = (2048u + (uint32_t)n) << 4;
  std::vector<uint32_t> ell2, ell3;
  if (packed) ell2.assign(total2 + 2 * 256, pad2);
  if (triangle) ell3.assign(total2 + 2 * 256, pad3);
  // One item deals a slice's entries for `ell` or one lane group of a slice
  // for a packed form; all are independent and run on the host's threads.
  // The searches take nearly all of the build's time: for 2583 strings of 29
  // orbitals (one thread for `ell`, one thread per slice for each packed form
  // in turn) that was 37 of 49 ms; with this split and the searches' pair sets
  // as bits the whole build takes 22 ms.
  const int ng = lane_groups(wide), forms = 1 + (packed ? ng : 0) + (triangle ? ng : 0);
  parallel_for(c, nsl * forms, [&](int item) {
    const int sl = item / forms, f = item % forms;
    auto each = [&](int l, auto take) {
      const uint32_t r = perm[(size_t)sl * 64 + l];
      if (r != 0xffffffffu)
        for (uint64_t k = off[r]; k < off[r + 1]; k++)
          take((uint32_t)(ent[k] & 0xffffffffull), (uint32_t)((ent[k] >> 32) & 0x7fffffffull), (uint32_t)(ent[k] >> 63));
    };
    if (f == 0) {
      std::vector<uint32_t> rows[64];
      for (int l = 0; l < 64; l++)
        each(l, [&](uint32_t ket, uint32_t pq, uint32_t neg) { rows[l].push_back(ket | (pq << 16) | (neg << 31)); });
      schedule_slice(rows, sl_len[sl], (uint32_t)c.K, (uint32_t)n, ell.data() + sl_off[sl]);
    } else if (f <= ng) {
      schedule_slice_packed(
          [&](int l, std::vector<uint32_t> &v) {
            each(l, [&](uint32_t ket, uint32_t pq, uint32_t neg) {
              v.push_back((((uint32_t)c.K + ket) << 4) | (pq << 19) | (neg << 31));
            });
          },
          f - 1, sl_len[sl], pad2, ell2.data() + sl_off2[sl], wide);
    } else {
      const uint32_t L = (uint32_t)c.L, Kt = (uint32_t)c.Kt;
      schedule_slice_packed(
          [&](int l, std::vector<uint32_t> &v) {
            each(l, [&](uint32_t ket, uint32_t pq, uint32_t neg) {
              const uint32_t a = pq / L, b = pq % L, hi = a > b ? a : b, lo = a > b ? b : a;
              v.push_back(((2048u + ket) << 4) | ((hi * (hi + 1) / 2 + lo + (neg ? Kt : 0u)) << 19));
            });
          },
          f - 1 - ng, sl_len[sl], pad3, ell3.data() + sl_off2[sl], wide);
    }
  });
  const StreamWait wait(c);
  auto put = [&](const void *src, size_t bytes) {
    void *dst = dalloc(c, bytes);
    SBDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c.stream));
    return dst;
  };
  t.nslice = nsl;
  t.ell = (uint32_t *)put(ell.data(), sizeof(uint32_t) * ell.size());
  t.perm = (uint32_t *)put(perm.data(), sizeof(uint32_t) * perm.size());
  t.sl_off = (uint64_t *)put(sl_off.data(), sizeof(uint64_t) * nsl);
  t.sl_len = (uint32_t *)put(sl_len.data(), sizeof(uint32_t) * nsl);
  if (triangle) {
    for (uint32_t &w : ell3) w = ((((w >> 4) & 0x7fffu) - 2048u) << 4) | (((w >> 19) & 0xfffu) << 21);
    t.ell3 = (uint32_t *)put(ell3.data(), sizeof(uint32_t) * ell3.size());
  }
  if (packed) {
    t.ell2 = (uint32_t *)put(ell2.data(), sizeof(uint32_t) * ell2.size());
    t.sl_off2 = (uint64_t *)put(sl_off2.data(), sizeof(uint64_t) * nsl);
    t.sl_len2 = (uint32_t *)put(sl_len2.data(), sizeof(uint32_t) * nsl);
  }
  SBDX_HIP(hipStreamSynchronize(c.stream));
  t.has_ell = true;
  t.has_ell2 = packed;
  t.has_ell3 = triangle;
}

// Ket-range parts of the sliced-ELL singles (SpinTables::pell): part p holds
// the entries with ket in [p*h, (p+1)*h), h = ceil(n/nparts), ket stored as
// ket - p*h, with the slices and row order of t.perm.
void build_singles_ell_parts(Context &c, SpinTables &t, int nparts) {
  if (!t.has_ell || nparts < 2 || t.nparts == nparts) return;
  const int n = t.n;
  const int h = (n + nparts - 1) / nparts;
  std::vector<uint64_t> off(n + 1), ent(t.ns);
  std::vector<uint32_t> perm((size_t)t.nslice * 64);
  SBDX_HIP(hipMemcpyAsync(off.data(), t.s_off, sizeof(uint64_t) * (n + 1), hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipMemcpyAsync(ent.data(), t.s_ent, sizeof(uint64_t) * t.ns, hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipMemcpyAsync(perm.data(), t.perm, sizeof(uint32_t) * perm.size(), hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipStreamSynchronize(c.stream));
  const uint32_t pad = (uint32_t)c.K << 16;
  t.pell.assign(nparts, nullptr);
  t.psl_off.assign(nparts, nullptr);
  t.psl_len.assign(nparts, nullptr);
  for (int p = 0; p < nparts; p++) {
    const uint64_t lo = (uint64_t)p * h, hi = std::min<uint64_t>((uint64_t)(p + 1) * h, (uint64_t)n);
    std::vector<uint32_t> sl_len(t.nslice);
    std::vector<uint64_t> sl_off(t.nslice);
    uint64_t total = 0;
    for (int s = 0; s < t.nslice; s++) {
      uint32_t mx = 0;
      for (int l = 0; l < 64; l++) {
        const uint32_t r = perm[(size_t)s * 64 + l];
        if (r == 0xffffffffu) continue;
        uint32_t cnt = 0;
        for (uint64_t e = off[r]; e < off[r + 1]; e++) {
          const uint64_t k = ent[e] & 0xffffffffull;
          cnt += (k >= lo && k < hi);
        }
        mx = std::max(mx, cnt);
      }
      sl_len[s] = mx;
      sl_off[s] = total;
      total += (uint64_t)mx * 64;
    }
    std::vector<uint32_t> ell(total + 1, pad);
    std::vector<uint32_t> rows[64];
    for (int s = 0; s < t.nslice; s++) {
      for (int l = 0; l < 64; l++) {
        rows[l].clear();
        const uint32_t r = perm[(size_t)s * 64 + l];
        if (r == 0xffffffffu) continue;
        for (uint64_t e = off[r]; e < off[r + 1]; e++) {
          const uint64_t ket = ent[e] & 0xffffffffull;
          if (ket < lo || ket >= hi) continue;
          const uint32_t pq = (uint32_t)((ent[e] >> 32) & 0x7fffffffull);
          rows[l].push_back((uint32_t)(ket - lo) | (pq << 16) | ((ent[e] >> 63) ? 0x80000000u : 0u));
        }
      }
      schedule_slice(rows, sl_len[s], (uint32_t)c.K, (uint32_t)(hi - lo), ell.data() + sl_off[s]);
    }
    t.pell[p] = (uint32_t *)dalloc(c, sizeof(uint32_t) * ell.size());
    t.psl_off[p] = (uint64_t *)dalloc(c, sizeof(uint64_t) * t.nslice);
    t.psl_len[p] = (uint32_t *)dalloc(c, sizeof(uint32_t) * t.nslice);
    SBDX_HIP(hipMemcpyAsync(t.pell[p], ell.data(), sizeof(uint32_t) * ell.size(), hipMemcpyHostToDevice, c.stream));
    SBDX_HIP(hipMemcpyAsync(t.psl_off[p], sl_off.data(), sizeof(uint64_t) * t.nslice, hipMemcpyHostToDevice, c.stream));
    SBDX_HIP(hipMemcpyAsync(t.psl_len[p], sl_len.data(), sizeof(uint32_t) * t.nslice, hipMemcpyHostToDevice, c.stream));
    SBDX_HIP(hipStreamSynchronize(c.stream));
  }
  t.nparts = nparts;
  t.part_h = h;
}

// Tables of the RDM's mixed term (SpinTables::ra_*, rc_*, pb).
//
// Singles come in blocks.  The strings k + u that share the string k with
// one electron less are singles of each other, all of them: in the set's
// singles matrix they are a dense block over the orbitals u, with the sign
// s_u s_v, s_u = (-1)^(electrons of k below u).  Each single (r, j) lies in
// exactly one such block, k = r & j.  A block of m members holds m (m - 1)
// ordered pairs and is a column of the matrix-core kernel, which costs its
// tiles of 16 orbitals squared (4 cycles of a CU per tile pair and alpha
// pair of strings); below kBlockWorth pairs per tile pair the entries one by
// one are as cheap (some 0.3 cycles each) and its singles are left over.
// What is left over is regrouped by the string K = r | j with one electron
// more (members K - u, sign -s_u s_v) into sets of members whose pairs are
// all left over, grown greedily from the member with the most partners; the
// rest goes to the entry table.  On a set of the Hartree-Fock string, its
// singles and doubles the first kind covers the moves of a particle, the
// second those of a hole.  A set may list a string more than once (rows that
// are alike but do not couple); its copies would share an orbital's place in
// a column, so blocks that hold such a pair stay in the entry table.
namespace {
constexpr int kBlockWorth = 12;

struct Member {
  uint64_t key;
  uint32_t str;
  uint8_t orb;
};
struct Column {
  uint64_t key;
  uint32_t first;  // members [first, first + m) of the owner's list
  uint16_t m;
  int8_t tile;  // the one tile of its members, or -1
  uint8_t hole;
};

inline uint64_t bit_reverse(uint64_t v) {
  uint64_t r = 0;
  for (int i = 0; i < 64; i++) r |= ((v >> i) & 1ull) << (63 - i);
  return r;
}
inline bool odd_below(uint64_t key, int orb) { return __builtin_popcountll(key & ((1ull << orb) - 1ull)) & 1; }
}  // namespace

// Tables of the mixed term's block kernel (SpinTables::bk_*).  Columns are
// the particle blocks of the note above, sorted by the bit-reversed string
// (the lowest orbitals, the hole pattern, first), so that consecutive
// columns have nearly the same orbitals; 16 of them make a task over the 16
// bk_mt orbitals most of their members use, and a member outside that list
// keeps its singles in the entry table.  A column costs tiles x steps matrix
// instructions per 16 columns and alpha single (4 cycles of a CU per tile,
// step and column in FP64); an ordered pair in the entry table some 0.15.
// They run on different units at the same time, so the line is drawn at
// kColWorth pairs per tile and step.
namespace {
constexpr int kColWorth = 4;
}

// The alpha set's tables: bk_order, bk_ent.
static void build_blocks_bra(Context &c, SpinTables &t, const std::vector<uint64_t> &strs) {
  const int n = t.n, L = c.L;
  std::vector<uint64_t> off, ent;
  download_singles(c, t, off, ent);
  // order of the bras: those with more than twice the average singles
  // first (the last blocks of a launch are then short), the rest by the
  // bit-reversed string, so that bras that run together share ket rows;
  // the 32 blocks that run on one XCD at a time get neighbours
  std::vector<uint32_t> ord(n);
  for (int i = 0; i < n; i++) ord[i] = (uint32_t)i;
  const double heavy = 2.0 * (double)t.ns / n;
  std::vector<uint64_t> rev(n);
  for (int i = 0; i < n; i++) rev[i] = bit_reverse(strs[i]);
  std::stable_sort(ord.begin(), ord.end(), [&](uint32_t a, uint32_t b) {
    const uint64_t la = off[a + 1] - off[a], lb = off[b + 1] - off[b];
    const bool ha = (double)la > heavy, hb = (double)lb > heavy;
    if (ha != hb) return ha;
    return ha ? la > lb : rev[a] < rev[b];
  });
  std::vector<uint32_t> blk(ord);
  for (int w = 0; w + 256 <= n; w += 256)
    for (int b = 0; b < 256; b++) blk[w + b] = ord[w + (b & 7) * 32 + (b >> 3)];
  std::vector<uint64_t> e2(t.ns + n);
  for (int r = 0; r < n; r++) {
    uint64_t *o = e2.data() + off[r] + r;
    for (uint64_t k = off[r]; k < off[r + 1]; k++) {
      const uint32_t pq = (uint32_t)((ent[k] >> 32) & 0x7fffffffull), a = pq / L, b = pq % L;
      const uint64_t tri = a > b ? a * (a + 1) / 2 + b : b * (b + 1) / 2 + a;
      *o++ = (ent[k] & 0xffffffffull) | (tri << 32) | (ent[k] & (1ull << 63));
    }
    *o = (uint64_t)r | (1ull << 62);
  }
  const StreamWait wait(c);
  auto put = [&](const void *src, size_t bytes) {
    void *dst = dalloc(c, bytes);
    if (bytes) SBDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c.stream));
    return dst;
  };
  t.bk_order = (uint32_t *)put(blk.data(), sizeof(uint32_t) * n);
  t.bk_ent = (uint64_t *)put(e2.data(), sizeof(uint64_t) * e2.size());
  SBDX_HIP(hipStreamSynchronize(c.stream));
}

// The beta set's tables; has_blk where the form holds them.
static void build_blocks_ket(Context &c, SpinTables &t, const std::vector<uint64_t> &strs) {
  const int n = t.n, L = c.L, Kt = c.Kt;
  t.has_blk = false;
  if (!c.eri_rs_sym || 2 * Kt + 1 > 2048) return;
  auto image = [&](int pb) { return ((size_t)2 * Kt + 1 + n + 1) << pb; };
  if (n < 8192 && image(4) <= c.lds_limit) t.bk_pb = 4;
  else if (n < 16384 && image(3) <= c.lds_limit) t.bk_pb = 3;
  else return;
  t.bk_mt = L <= 16 ? 1 : 2;
  const int MT = t.bk_mt;
  std::vector<uint64_t> off, ent;
  download_singles(c, t, off, ent);
  // ---- columns
  std::vector<Member> pm;
  pm.reserve((size_t)n * 16);
  for (int r = 0; r < n; r++)
    for (uint64_t o = strs[r]; o; o &= o - 1) {
      const int u = __builtin_ctzll(o);
      pm.push_back({strs[r] ^ (1ull << u), (uint32_t)r, (uint8_t)u});
    }
  std::sort(pm.begin(), pm.end(), [](const Member &a, const Member &b) {
    return a.key < b.key || (a.key == b.key && a.orb < b.orb);
  });
  auto worth = [&](int m) { return m > 1 && m * (m - 1) >= kColWorth * MT * 4 * MT; };
  struct Col {
    uint64_t rev;
    uint32_t first, m;
  };
  std::vector<Col> cols;
  for (size_t i = 0; i < pm.size();) {
    size_t j = i;
    bool twice = false;  // two members at one orbital
    for (; j < pm.size() && pm[j].key == pm[i].key; j++) twice |= j > i && pm[j].orb == pm[j - 1].orb;
    if (!twice && worth((int)(j - i))) cols.push_back({bit_reverse(pm[i].key), (uint32_t)i, (uint32_t)(j - i)});
    i = j;
  }
  std::sort(cols.begin(), cols.end(), [](const Col &a, const Col &b) { return a.rev < b.rev; });
  // ---- tasks
  const int ntask = (int)((cols.size() + 15) / 16);
  auto tri = [](int a, int b) { return a > b ? a * (a + 1) / 2 + b : b * (b + 1) / 2 + a; };
  std::vector<uint32_t> step(1, 0u);
  std::vector<uint2> tab;
  const uint2 none = make_uint2((uint32_t)(2 * Kt) * 0x00010001u, (uint32_t)n);
  // column of string r with the electron in u removed, where it is a member
  std::vector<int32_t> col_of((size_t)n * L, -1);
  // every string's accumulators: task, element | sign << 15
  std::vector<std::vector<std::pair<int, uint16_t>>> pos_of(n);
  for (int k = 0; k < ntask; k++) {
    const size_t c0 = (size_t)16 * k, c1 = std::min(cols.size(), c0 + 16);
    int use[64] = {};
    for (size_t q = c0; q < c1; q++)
      for (uint32_t i = 0; i < cols[q].m; i++) use[pm[cols[q].first + i].orb]++;
    std::vector<int> list;
    for (int u = 0; u < L; u++)
      if (use[u]) list.push_back(u);
    std::stable_sort(list.begin(), list.end(), [&](int a, int b) { return use[a] > use[b]; });
    if ((int)list.size() > 16 * MT) list.resize(16 * MT);
    std::sort(list.begin(), list.end());
    int pos[64];
    std::fill(pos, pos + 64, -1);
    for (size_t i = 0; i < list.size(); i++) pos[list[i]] = (int)i;
    const int nu = (int)list.size();
    const size_t s0 = tab.size() / 64;
    const int ns = 2 * ((nu + 7) / 8);  // the kernel takes two at a time
    step.push_back((uint32_t)(s0 + ns));
    tab.resize(tab.size() + (size_t)64 * ns, none);
    for (int iv = 0; iv < nu; iv++)
      for (int iu = 0; iu < nu; iu++) {
        if (iu == iv) continue;
        uint32_t &w = tab[(s0 + iv / 4) * 64 + 16 * (iv % 4) + iu % 16].x;
        const int sh = 16 * (iu / 16);
        w = (w & ~(0xffffu << sh)) | ((uint32_t)tri(list[iu], list[iv]) << sh);
      }
    for (size_t q = c0; q < c1; q++)
      for (uint32_t i = 0; i < cols[q].m; i++) {
        const Member &mb = pm[cols[q].first + i];
        const int p = pos[mb.orb], cc = (int)(q - c0);
        if (p < 0) continue;
        const uint32_t v = mb.str | (odd_below(mb.key, mb.orb) ? 0x8000u : 0u);
        tab[(s0 + p / 4) * 64 + 16 * (p % 4) + cc].y = v;
        pos_of[mb.str].push_back({k, (uint16_t)(p * 16 + cc + ((v & 0x8000u) ? 0x8000u : 0u))});
        col_of[(size_t)mb.str * L + mb.orb] = (int32_t)q;
      }
  }
  t.bk_ntask = ntask;
  // at the end a group's LDS holds a sum per string and, behind them, the
  // accumulators of as many tasks at a time as its image has room for (more
  // room is taken where one block fills a CU's LDS anyway)
  const size_t unit = (size_t)MT * 256 * 8, sums = (size_t)8 * n;
  size_t room = image(t.bk_pb);
  if (room * 2 > c.lds_limit) room = c.lds_limit;
  room = std::max(room, sums + unit);
  t.bk_tp = (int)std::max<size_t>(1, std::min<size_t>({(room - sums) / unit, (size_t)std::max(ntask, 1), size_t{20}}));
  t.bk_image = (std::max(image(t.bk_pb), sums + t.bk_tp * unit) + 15) / 16 * 16;
  if (t.bk_image > c.lds_limit) return;
  const int npass = (ntask + t.bk_tp - 1) / t.bk_tp;
  std::vector<uint32_t> col_off;
  std::vector<uint16_t> col_pos;
  for (int q = 0; q < npass; q++) {
    for (int r = 0; r < n; r++) {
      col_off.push_back((uint32_t)col_pos.size());
      for (const auto &v : pos_of[r])
        if (v.first / t.bk_tp == q)
          col_pos.push_back((uint16_t)(v.second + (v.first % t.bk_tp) * MT * 256));
    }
    col_off.push_back((uint32_t)col_pos.size());
  }
  t.bk_nstep = (int)step.back();
  tab.resize(tab.size() + 6 * 64, none);  // the kernel loads up to four steps ahead
  // ---- the rest, entry by entry
  auto covered = [&](int r, uint64_t e) {
    const uint32_t pq = (uint32_t)((e >> 32) & 0x7fffffffull);
    const int32_t a = col_of[(size_t)r * L + pq / L];
    return a >= 0 && a == col_of[(e & 0xffffffffull) * L + pq % L];
  };
  std::vector<uint32_t> cnt(n, 0);
  size_t nrest = 0;
  for (int r = 0; r < n; r++) {
    for (uint64_t k = off[r]; k < off[r + 1]; k++) cnt[r] += covered(r, ent[k]) ? 0 : 1;
    nrest += cnt[r];
  }
  // the reference string, when the rows differ from it in fewer orbitals
  // than they have electrons
  size_t nd = 0, ne = 0;
  for (int r = 0; r < n; r++) {
    nd += __builtin_popcountll(strs[r] ^ strs[0]);
    ne += __builtin_popcountll(strs[r]);
  }
  t.bk_ref = nd < ne ? strs[0] : 0ull;
  std::vector<uint32_t> order(n);
  for (int i = 0; i < n; i++) order[i] = (uint32_t)i;
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) {
    const uint32_t ga = (cnt[a] + 3) / 4, gb = (cnt[b] + 3) / 4;
    if (ga != gb) return ga > gb;
    return __builtin_popcountll(strs[a] ^ t.bk_ref) > __builtin_popcountll(strs[b] ^ t.bk_ref);
  });
  const int nsl = (n + 63) / 64;
  std::vector<uint32_t> perm((size_t)nsl * 64, (uint32_t)n), soff(nsl), len(nsl);
  int most = 0;  // orbitals in which a row differs from the reference
  for (int r = 0; r < n; r++) most = std::max(most, __builtin_popcountll(strs[r] ^ t.bk_ref));
  t.bk_nrec = (most + 8) / 8;
  std::vector<uint16_t> rec((size_t)nsl * t.bk_nrec * 64 * 8, (uint16_t)(2 * Kt));
  uint32_t tot = 0;
  for (int sl = 0; sl < nsl; sl++) {
    uint32_t mx = 0, md = 0;
    for (int l = 0; l < 64; l++) rec[((size_t)sl * t.bk_nrec * 64 + l) * 8] = (uint16_t)n;
    for (int l = 0; l < 64 && sl * 64 + l < n; l++) {
      const uint32_t r = order[(size_t)sl * 64 + l];
      perm[(size_t)sl * 64 + l] = r;
      mx = std::max(mx, (cnt[r] + 3) / 4);
      rec[((size_t)sl * t.bk_nrec * 64 + l) * 8] = (uint16_t)r;
      uint32_t q = 1;
      for (uint64_t o = strs[r] ^ t.bk_ref; o; o &= o - 1, q++) {
        const int k = __builtin_ctzll(o);
        rec[(((size_t)sl * t.bk_nrec + q / 8) * 64 + l) * 8 + q % 8] =
            (uint16_t)(k * (k + 3) / 2 + (((t.bk_ref >> k) & 1ull) ? Kt : 0));
      }
      md = std::max(md, q - 1);
    }
    soff[sl] = tot;
    len[sl] = mx | (md << 16);
    tot += mx;
  }
  t.bk_nslice = nsl;
  t.bk_ngroup = (int)tot;
  if (!blk_worth(c, t.ns - nrest)) return;
  // all tables of the form, the bras' and those of blk_tables among them
  const size_t bytes = sizeof(uint32_t) * (col_off.size() + step.size() + perm.size() + 2 * (size_t)nsl + c.na +
                                           (size_t)(tot + 4) * 256) +
                       sizeof(uint16_t) * (col_pos.size() + rec.size()) + sizeof(uint2) * tab.size() +
                       sizeof(uint64_t) * (c.A.ns + c.na) + sizeof(double) * Kt * ((size_t)Kt + 1 + c.na);
  size_t free_b = 0, total_b = 0;
  SBDX_HIP(hipMemGetInfo(&free_b, &total_b));
  if (bytes >= free_b / 4) return;  // the room may be wanted for a solver's basis
  // dealt in the word layout of schedule_slice_packed, whose fields hold LDS
  // elements: the ket's 2 Kt + 1 + ket, the ERI value's triangle index
  const uint32_t xe = 2u * (uint32_t)Kt + 1u;
  std::vector<uint32_t> ell((size_t)(tot + 4) * 256);
  const uint32_t pad = (xe + (uint32_t)n) << 4;
  std::fill(ell.begin(), ell.end(), (uint32_t)n << t.bk_pb);
  const bool wide = t.bk_pb == 4;
  const int ng = lane_groups(wide);
  parallel_for(c, nsl * ng, [&](int item) {
    const int sl = item / ng;
    const size_t words = (size_t)(len[sl] & 0xffffu) * 256;
    std::vector<uint32_t> dealt(words, pad);
    uint32_t longest = 0;
    auto rows = [&](int l, std::vector<uint32_t> &v) {
      const uint32_t r = perm[(size_t)sl * 64 + l];
      if (r == (uint32_t)n) return;
      for (uint64_t k = off[r]; k < off[r + 1]; k++) {
        if (covered((int)r, ent[k])) continue;
        const uint32_t pq = (uint32_t)((ent[k] >> 32) & 0x7fffffffull);
        const uint32_t w = (uint32_t)tri((int)(pq / L), (int)(pq % L)) + ((ent[k] >> 63) ? (uint32_t)Kt : 0u);
        v.push_back(((xe + (uint32_t)(ent[k] & 0xffffffffull)) << 4) | (w << 19));
      }
    };
    for (int l = 0; l < 64; l++) {
      const uint32_t r = perm[(size_t)sl * 64 + l];
      if (r != (uint32_t)n) longest = std::max(longest, cnt[r]);
    }
    schedule_slice_packed(rows, item % ng, longest, pad, dealt.data(), wide);
    // repacked lane by lane: a padding word stays as `ell` was filled
    uint32_t *o = ell.data() + (size_t)soff[sl] * 256;
    for (size_t i = 0; i < words; i++)
      if (dealt[i] != pad) o[i] = ((((dealt[i] >> 4) & 0x7fffu) - xe) << t.bk_pb) | ((dealt[i] >> 19) << 21);
  });
  const StreamWait wait(c);
  auto put = [&](const void *src, size_t bytes) {
    void *dst = dalloc(c, bytes);
    if (bytes) SBDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c.stream));
    return dst;
  };
  t.bk_col_off = (uint32_t *)put(col_off.data(), sizeof(uint32_t) * col_off.size());
  t.bk_col_pos = (uint16_t *)put(col_pos.data(), sizeof(uint16_t) * col_pos.size());
  t.bk_step = (uint32_t *)put(step.data(), sizeof(uint32_t) * step.size());
  t.bk_tab = (uint2 *)put(tab.data(), sizeof(uint2) * tab.size());
  t.bk_perm = (uint32_t *)put(perm.data(), sizeof(uint32_t) * perm.size());
  t.bk_rec = (uint4 *)put(rec.data(), sizeof(uint16_t) * rec.size());
  t.bk_off = (uint32_t *)put(soff.data(), sizeof(uint32_t) * nsl);
  t.bk_len = (uint32_t *)put(len.data(), sizeof(uint32_t) * nsl);
  t.bk_ell = (uint32_t *)put(ell.data(), sizeof(uint32_t) * ell.size());
  SBDX_HIP(hipStreamSynchronize(c.stream));
  t.has_blk = true;
}

// On a context's first FP64 product: one for FP32 or symmetric products,
// density matrices or the diagonal needs none of this.
void build_blocks(Context &c) {
  build_blocks_ket(c, c.B, c.h_bstr);
  if (c.B.has_blk) build_blocks_bra(c, c.A, c.h_astr);
}

// Gives back what build_blocks has laid down.
void release_blocks(Context &c) {
  auto drop = [&](auto *&p) {
    dfree(c, p);
    p = nullptr;
  };
  c.B.has_blk = false;
  for (SpinTables *t : {&c.A, &c.B}) {
    drop(t->bk_ent), drop(t->bk_order);
    drop(t->bk_col_off), drop(t->bk_col_pos), drop(t->bk_step), drop(t->bk_tab);
    drop(t->bk_perm), drop(t->bk_rec), drop(t->bk_off), drop(t->bk_len), drop(t->bk_ell);
  }
}

void build_rdm_tables(Context &c, SpinTables &t, const std::vector<uint64_t> &strs, bool as_alpha, bool as_beta) {
  const int n = t.n, L = c.L;
  const size_t K = (size_t)c.K;
  std::vector<uint64_t> off, ent;
  download_singles(c, t, off, ent);
  auto put = [&](void *&dst, const void *src, size_t bytes) {
    dst = dalloc(c, bytes);
    if (bytes) SBDX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, c.stream));
  };
  std::vector<uint64_t> aent;
  std::vector<uint4> items;
  const StreamWait wait_a(c);
  if (as_alpha) {
    std::vector<size_t> cnt(K + 1, 0);
    auto kept = [&](uint64_t e) {
      const uint32_t pq = (uint32_t)((e >> 32) & 0x7fffffffull);
      return pq / L > pq % L ? (int)pq : -1;
    };
    for (size_t k = 0; k < t.ns; k++) {
      const int pq = kept(ent[k]);
      if (pq >= 0) cnt[pq + 1]++;
    }
    for (int r = 0; r < n; r++)
      for (uint64_t o = strs[r]; o; o &= o - 1) cnt[(size_t)__builtin_ctzll(o) * (L + 1) + 1]++;
    for (size_t i = 0; i < K; i++) cnt[i + 1] += cnt[i];
    std::vector<size_t> at(cnt.begin(), cnt.end() - 1);
    aent.resize(cnt[K]);
    for (int r = 0; r < n; r++) {
      for (uint64_t k = off[r]; k < off[r + 1]; k++) {
        const int pq = kept(ent[k]);
        if (pq >= 0)
          aent[at[pq]++] = (uint64_t)r | ((ent[k] & 0x7fffffffull) << 32) | (ent[k] & (1ull << 63));
      }
      for (uint64_t o = strs[r]; o; o &= o - 1)
        aent[at[(size_t)__builtin_ctzll(o) * (L + 1)]++] = (uint64_t)r | ((uint64_t)r << 32);
    }
    // items of equal length: long ones amortize the sums over the block and
    // the atomics at an item's end, short ones keep every CU busy (at least
    // eight items per CU)
    const size_t len = std::min<size_t>(32, std::max<size_t>(1, aent.size() / ((size_t)8 * c.n_cu)));
    for (size_t i = 0; i < K; i++)
      for (size_t e = cnt[i]; e < cnt[i + 1]; e += len)
        items.push_back(make_uint4((unsigned)i, (unsigned)e, (unsigned)std::min(e + len, cnt[i + 1]), 0u));
    t.ra_nitem = (int)items.size();
    void *p;
    put(p, aent.data(), sizeof(uint64_t) * aent.size());
    t.ra_ent = (uint64_t *)p;
    put(p, items.data(), sizeof(uint4) * items.size());
    t.ra_item = (uint4 *)p;
  }
  t.rc_nrange = 0;
  t.pb_nslice = 0;
  if (!as_beta || n >= 32767) {
    SBDX_HIP(hipStreamSynchronize(c.stream));
    return;
  }
  // particle blocks: (string, removed orbital) sorted by the remainder
  std::vector<Member> pm;
  pm.reserve((size_t)n * 16);
  for (int r = 0; r < n; r++)
    for (uint64_t o = strs[r]; o; o &= o - 1) {
      const int u = __builtin_ctzll(o);
      pm.push_back({strs[r] ^ (1ull << u), (uint32_t)r, (uint8_t)u});
    }
  std::sort(pm.begin(), pm.end(), [](const Member &a, const Member &b) {
    return a.key < b.key || (a.key == b.key && a.orb < b.orb);
  });
  std::vector<Column> cols;
  std::vector<uint64_t> big((size_t)n, 0);  // bit u of big[r]: r - u is the remainder of a kept block
  const int nt = (L + 15) / 16;
  auto tile_of = [](uint32_t tiles) { return (tiles & (tiles - 1)) ? -1 : __builtin_ctz(tiles); };
  auto worth = [&](int m, int tile) {
    const int q = tile < 0 ? nt : 1;
    return m > 1 && m * (m - 1) >= kBlockWorth * q * q;
  };
  for (size_t i = 0; i < pm.size();) {
    size_t j = i;
    uint32_t tiles = 0;
    bool twice = false;
    for (; j < pm.size() && pm[j].key == pm[i].key; j++) {
      tiles |= 1u << (pm[j].orb >> 4);
      twice |= j > i && pm[j].orb == pm[j - 1].orb;
    }
    if (!twice && worth((int)(j - i), tile_of(tiles))) {
      for (size_t k = i; k < j; k++) big[pm[k].str] |= 1ull << pm[k].orb;
      cols.push_back({pm[i].key, (uint32_t)i, (uint16_t)(j - i), (int8_t)tile_of(tiles), 0});
    }
    i = j;
  }
  // what they leave over, by r | j: entry indices with their missing orbital
  struct Left {
    uint64_t key;
    uint32_t ent, str;
    uint8_t miss, add;  // r = K - miss, j = K - add
  };
  std::vector<Left> left;
  for (int r = 0; r < n; r++)
    for (uint64_t k = off[r]; k < off[r + 1]; k++) {
      const uint32_t pq = (uint32_t)((ent[k] >> 32) & 0x7fffffffull);
      const int p = pq / L, q = pq % L;
      if (!((big[r] >> p) & 1ull))
        left.push_back({strs[r] | (1ull << q), (uint32_t)k, (uint32_t)r, (uint8_t)q, (uint8_t)p});
    }
  std::sort(left.begin(), left.end(), [](const Left &a, const Left &b) {
    return a.key < b.key || (a.key == b.key && a.ent < b.ent);
  });
  std::vector<Member> hm;
  std::vector<uint8_t> done(left.size(), 0);
  for (size_t i = 0; i < left.size();) {
    size_t j = i;
    uint64_t adj[64] = {}, verts = 0;
    uint32_t who[64] = {};
    bool twice = false;
    for (; j < left.size() && left[j].key == left[i].key; j++) {
      const int v = left[j].miss;
      twice |= ((verts >> v) & 1ull) && who[v] != left[j].str;
      adj[v] |= 1ull << left[j].add;
      verts |= 1ull << v;
      who[v] = left[j].str;
    }
    if (twice) verts = 0;
    int cls[64];
    std::fill(cls, cls + 64, -1);
    for (int nc = 0;; nc++) {
      auto best = [&](uint64_t among) {  // the member with the most partners among `among`
        int b = -1, bd = -1;
        for (uint64_t o = among; o; o &= o - 1) {
          const int v = __builtin_ctzll(o), dg = __builtin_popcountll(adj[v] & among);
          if (dg > bd) b = v, bd = dg;
        }
        return b;
      };
      const int v0 = best(verts);
      if (v0 < 0) break;
      uint64_t set = 1ull << v0, cand = adj[v0] & verts;
      while (cand) {
        const int v = best(cand);
        set |= 1ull << v;
        cand &= adj[v];
      }
      uint32_t tiles = 0;
      for (uint64_t o = set; o; o &= o - 1) tiles |= 1u << (__builtin_ctzll(o) >> 4);
      if (!worth(__builtin_popcountll(set), tile_of(tiles))) break;
      cols.push_back(
          {left[i].key, (uint32_t)hm.size(), (uint16_t)__builtin_popcountll(set), (int8_t)tile_of(tiles), 1});
      for (uint64_t o = set; o; o &= o - 1) {
        const int v = __builtin_ctzll(o);
        hm.push_back({left[i].key, who[v], (uint8_t)v});
        cls[v] = nc;
      }
      verts &= ~set;
    }
    for (size_t k = i; k < j; k++) done[k] = cls[left[k].miss] >= 0 && cls[left[k].miss] == cls[left[k].add];
    i = j;
  }
  // columns of one kind and tile together, each run padded to steps of 4
  for (auto &cl : cols) cl.key = bit_reverse(cl.key);
  std::sort(cols.begin(), cols.end(), [](const Column &a, const Column &b) {
    if (a.hole != b.hole) return a.hole < b.hole;
    if (a.tile != b.tile) return a.tile < b.tile;
    return a.key < b.key;
  });
  std::vector<uint64_t> tab;
  const uint64_t none = (uint64_t)n * 0x0001000100010001ull;
  for (size_t i = 0; i < cols.size();) {
    size_t j = i;
    while (j < cols.size() && cols[j].hole == cols[i].hole && cols[j].tile == cols[i].tile) j++;
    const int s0 = (int)(tab.size() / 64), ns = (int)((j - i + 3) / 4);
    tab.resize(tab.size() + (size_t)64 * ns, none);
    for (size_t k = i; k < j; k++) {
      const Member *mb = (cols[k].hole ? hm.data() : pm.data()) + cols[k].first;
      uint64_t *w = tab.data() + (size_t)64 * (s0 + (k - i) / 4) + 16 * ((k - i) % 4);
      for (int q = 0; q < cols[k].m; q++) {
        const int u = mb[q].orb, sh = 16 * (u >> 4);
        const uint64_t v = mb[q].str | (odd_below(mb[q].key, u) ? 0x8000ull : 0ull);
        w[u & 15] = (w[u & 15] & ~(0xffffull << sh)) | (v << sh);
      }
    }
    if (t.rc_nrange >= 24) throw Error(3, "rdm tables: too many kinds of columns");
    t.rc_range[t.rc_nrange++] = make_int4(s0, s0 + ns, cols[i].tile, cols[i].hole);
    i = j;
  }
  // the entry table of the rest: every pair's entries in runs of at most
  // `run`, some of the shortest for which a round of slices (8, one per
  // wavefront) or a few hold all runs: half as many again as there are pairs
  // with entries, so that long pairs are split among the others' lanes.  With
  // one round for any number of pairs, more than 512 of them stayed whole, and
  // a wavefront with the longest ones held up the rest: density matrices of
  // 1500 x 8000 strings drawn over 40 orbitals 21 ms, 12 with these runs, of
  // the Hartree-Fock string's excitations 12.6 and 9.4; 1500 x 4001 over 36
  // orbitals 7.8 and 5.9.
  std::vector<std::vector<uint32_t>> bin(K);
  size_t nrest = 0;
  for (size_t k = 0; k < left.size(); k++) {
    if (done[k]) continue;
    const uint64_t e = ent[left[k].ent];
    bin[(e >> 32) & 0x7fffffffull].push_back(left[k].str | ((uint32_t)(e & 0x7fffull) << 15) |
                                             ((uint32_t)(e >> 63) << 31));
    nrest++;
  }
  auto runs_of = [&](size_t len) {
    size_t q = 0;
    for (const auto &v : bin) q += (v.size() + len - 1) / len;
    return q;
  };
  const size_t pairs = runs_of(nrest + 1), most = std::max<size_t>(512, (pairs + pairs / 2 + 511) / 512 * 512);
  size_t run = std::max<size_t>(4, (nrest + most - 1) / most);
  while (runs_of(run) > most) run += (run + 7) / 8;
  struct Run {
    uint32_t pair, first, len;
  };
  std::vector<Run> runs;
  for (size_t i = 0; i < K; i++)
    for (size_t k = 0; k < bin[i].size(); k += run)
      runs.push_back({(uint32_t)i, (uint32_t)k, (uint32_t)std::min(run, bin[i].size() - k)});
  std::stable_sort(runs.begin(), runs.end(), [](const Run &a, const Run &b) { return a.len > b.len; });
  const size_t nsl = (runs.size() + 63) / 64;
  std::vector<uint32_t> perm(nsl * 64, 0xffffffffu), len(nsl);
  std::vector<uint64_t> soff(nsl);
  std::vector<uint32_t> pb;
  for (size_t i = 0; i < runs.size(); i++) {
    if (i % 64 == 0) {
      soff[i / 64] = pb.size();
      len[i / 64] = runs[i].len;
      pb.resize(pb.size() + (size_t)64 * runs[i].len, (uint32_t)n | ((uint32_t)n << 15));
    }
    perm[i] = runs[i].pair;
    for (uint32_t k = 0; k < runs[i].len; k++) pb[soff[i / 64] + 64 * k + i % 64] = bin[runs[i].pair][runs[i].first + k];
  }
  const StreamWait wait_b(c);
  void *p;
  put(p, tab.data(), sizeof(uint64_t) * tab.size());
  t.rc_tab = (uint64_t *)p;
  put(p, pb.data(), sizeof(uint32_t) * pb.size());
  t.pb = (uint32_t *)p;
  put(p, soff.data(), sizeof(uint64_t) * nsl);
  t.pb_off = (uint64_t *)p;
  put(p, len.data(), sizeof(uint32_t) * nsl);
  t.pb_len = (uint32_t *)p;
  put(p, perm.data(), sizeof(uint32_t) * perm.size());
  t.pb_perm = (uint32_t *)p;
  t.pb_nslice = (int)nsl;
  SBDX_HIP(hipStreamSynchronize(c.stream));
}

void compute_diag(Context &c) {
  const unsigned nchunk = cdiv(c.nb, 256);
  ProfScope ps(c, "diag");
  hipLaunchKernelGGL(k_diag, dim3((unsigned)(c.na * nchunk)), dim3(256), 0, c.stream, (int)c.nb,
                     (int)nchunk, c.L, c.I0, (c.B.alias && c.na == c.nb) ? 1 : 0, c.B.str, c.A.e1, c.B.e1,
                     c.A.jsum, c.hii);
  check_launch("k_diag");
}

void sign_convert(Context &c, const double *in, double *out) {
  const unsigned nchunk = cdiv(c.nb, 256);
  ProfScope ps(c, "sign");
  hipLaunchKernelGGL(k_sign<false>, dim3((unsigned)(c.na * nchunk)), dim3(256), 0, c.stream,
                     (int)c.nb, (int)nchunk, c.A.str, c.B.str, in, out);
  check_launch("k_sign");
}

void sign_convert_noprof(Context &c, const double *in, double *out) {
  const unsigned nchunk = cdiv(c.nb, 256);
  hipLaunchKernelGGL(k_sign<false>, dim3((unsigned)(c.na * nchunk)), dim3(256), 0, c.stream,
                     (int)c.nb, (int)nchunk, c.A.str, c.B.str, in, out);
  check_launch("k_sign");
}

void sign_convert_add(Context &c, const double *in, double *out) {
  const unsigned nchunk = cdiv(c.nb, 256);
  ProfScope ps(c, "sign");
  hipLaunchKernelGGL(k_sign<true>, dim3((unsigned)(c.na * nchunk)), dim3(256), 0, c.stream,
                     (int)c.nb, (int)nchunk, c.A.str, c.B.str, in, out);
  check_launch("k_sign");
}

}  // namespace sbdx
