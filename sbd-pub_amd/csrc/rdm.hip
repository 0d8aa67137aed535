// 1-/2-RDM, chemistry/tpb/correlation.h:378-662 with the element rules of
// chemistry/basic/correlation.h:16-229 (ZeroDiff/OneDiff/TwoDiffCorrelation).
//
// Layout: one[s*L^2 + i + L*j], two[(s+2t)*L^4 + i + L*j + L^2*k + L^3*l].
// Work is done on the alpha-first vector W' = S*W: every contribution of the
// reference, w_bra*w_ket*(interleaved sign), equals w'_bra*w'_ket times the
// one-spin table sign (alpha single, beta single, or their product for the
// mixed term), so the per-pair sums below factor over the other spin:
//   same spin -> dots of the rows of w' (strings of this spin): rho[I] =
//                <I|I>, G[I,J] per single and double pair of strings
//   two spins -> T[pq][rs] = sum over the alpha pairs (I, J) of pq and the
//                beta pairs (i, j) of rs of s_a s_b w'[I,i] w'[J,j], where the
//                pairs of an orbital with itself (p == q: I = J with p
//                occupied) stand for the occupation numbers; then placed with
//                the reference's spin-orbital ordering rules.
#include <memory>
#include <mutex>
#include <string>

#include "common.h"

namespace sbdx {

typedef double d4 __attribute__((ext_vector_type(4)));
static inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

__device__ __forceinline__ double parity1r(uint64_t s, int a, int b) {
  int lo = a < b ? a : b, hi = a < b ? b : a;
  uint64_t mask = ((1ull << hi) - 1ull) ^ ((1ull << lo) - 1ull);
  int n = __popcll(s & mask) + (int)((s >> lo) & 1ull);
  return (n & 1) ? -1.0 : 1.0;
}

__device__ __forceinline__ double blk_sum256(double v, double *sh) {
  const int t = threadIdx.x;
  sh[t] = v;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) sh[t] += sh[t + s];
    __syncthreads();
  }
  const double r = sh[0];
  __syncthreads();
  return r;
}

__device__ __forceinline__ int row_of(const uint64_t *off, int n, uint64_t e) {
  int lo = 0, hi = n;  // off[lo] <= e < off[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (off[mid] <= e) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Per row r of w (rows x M): rho[r] = sum_m w^2
__global__ void __launch_bounds__(256) k_rdm_diag_rows(int M, const double *__restrict__ w,
                                                       double *__restrict__ rho) {
  __shared__ double sh[256];
  const int r = blockIdx.x;
  double s = 0.0;
  for (int m = threadIdx.x; m < M; m += 256) {
    const double v = w[(size_t)r * M + m];
    s += v * v;
  }
  const double t = blk_sum256(s, sh);
  if (threadIdx.x == 0) rho[r] = t;
}

// Same-spin ZeroDiff of one spin: rho[r * rstride] weights string r.
// one[p,p] += rho n_p and, for p != r, two[p,r,p,r] += rho n_p n_r and
// two[p,r,r,p] -= the same.  A wavefront walks kDiagStr strings, lane = r;
// the sums over the strings are collected in LDS (no two lanes of a
// wavefront share an element).  A wavefront loads its strings and weights at
// once, one a lane: one after the other they were most of the kernel's time,
// 24 us at 500 strings, 15 this way.
constexpr int kDiagStr = 32;
__global__ void __launch_bounds__(256) k_rdm_diag_pairs(int n, int L, int spin, const uint64_t *__restrict__ str,
                                                        const double *__restrict__ rho, size_t rstride,
                                                        double *__restrict__ one, double *__restrict__ two) {
  extern __shared__ double lds[];  // [L][L]
  const int L2 = L * L;
  for (int i = threadIdx.x; i < L2; i += 256) lds[i] = 0.0;
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int r0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * kDiagStr;
  static_assert(kDiagStr <= 64, "a lane holds one string");
  const int rl = r0 + lane;
  const bool has = lane < kDiagStr && rl < n;
  const uint64_t my_str = has ? str[rl] : 0;
  const double my_rho = has ? rho[(size_t)rl * rstride] : 0.0;
  for (int k = 0; k < kDiagStr && r0 + k < n; k++) {
    const uint64_t s = (uint64_t)__shfl((unsigned long long)my_str, k, 64);
    const double v = __shfl(my_rho, k, 64);
    if ((s >> lane) & 1ull)
      for (uint64_t o = s; o; o &= o - 1) atomicAdd(&lds[(__ffsll((unsigned long long)o) - 1) * L + lane], v);
  }
  __syncthreads();
  const size_t K = (size_t)L2, bs = (size_t)(3 * spin) * K * K;
  for (int i = threadIdx.x; i < L2; i += 256) {
    const double v = lds[i];
    if (v == 0.0) continue;
    const size_t p = i / L, r = i % L;
    if (p == r) {
      atomicAdd(&one[spin * K + p + L * p], v);
    } else {
      atomicAdd(&two[bs + p + L * r + K * (p + L * r)], v);
      atomicAdd(&two[bs + p + L * r + K * (r + L * p)], -v);
    }
  }
}

// Single pairs of one spin, e0 <= e < e1: out[e - e0] = s * sum_m w[I,m] w[J,m]
__global__ void __launch_bounds__(256) k_rdm_single_pairs(int n, int M, uint64_t e0, uint64_t e1,
                                                          const uint64_t *__restrict__ s_off,
                                                          const uint64_t *__restrict__ s_ent,
                                                          const double *__restrict__ w,
                                                          double *__restrict__ out) {
  __shared__ double sh[256];
  for (uint64_t e = e0 + blockIdx.x; e < e1; e += gridDim.x) {
    const int I = row_of(s_off, n, e);
    const uint64_t ent = s_ent[e];
    const size_t J = (uint32_t)(ent & 0xffffffffull);
    double s = 0.0;
    for (int m = threadIdx.x; m < M; m += 256) s += w[(size_t)I * M + m] * w[J * M + m];
    const double t = blk_sum256(s, sh);
    if (threadIdx.x == 0) out[e - e0] = (ent >> 63) ? -t : t;
  }
}

// Double pairs of one spin, e0 <= e < e1: out[e - e0] = sign * sum_m w[I,m] w[J,m]
__global__ void __launch_bounds__(256) k_rdm_double_pairs(int n, int M, uint64_t e0, uint64_t e1,
                                                          const uint64_t *__restrict__ d_off,
                                                          const uint32_t *__restrict__ d_ket,
                                                          const uint32_t *__restrict__ d_orb,
                                                          const uint64_t *__restrict__ str,
                                                          const double *__restrict__ w,
                                                          double *__restrict__ out) {
  __shared__ double sh[256];
  for (uint64_t e = e0 + blockIdx.x; e < e1; e += gridDim.x) {
  const int I = row_of(d_off, n, e);
  const size_t J = d_ket[e];
  double s = 0.0;
  for (int m = threadIdx.x; m < M; m += 256) s += w[(size_t)I * M + m] * w[J * M + m];
  const double t = blk_sum256(s, sh);
  if (threadIdx.x == 0) {
    const uint32_t o = d_orb[e];
    const int i = o & 255, j = (o >> 8) & 255, a = (o >> 16) & 255, b = (o >> 24) & 255;
    const uint64_t bra = str[I];
    double sg = parity1r(bra, i, a) * parity1r(bra, j, b);
    if (a > j || b < i) sg = -sg;
    out[e - e0] = sg * t;
  }
  }
}

// The Gram matrix G = w w^T of n rows of M values, its lower triangle (tiles
// across the diagonal whole).  A wave holds 16 T x 16 T elements over all
// columns, a block 2 x 2 waves (KS 1); or half the columns, a block two tiles
// side by side and their sums added in LDS (KS 2: for few rows, where whole
// tiles would leave SIMDs idle).  Operands come straight from memory into
// registers, PD - 1 stages of 8 columns ahead: lane group g of both operands
// takes columns 2 g and 2 g + 1 (a 16-byte load per row) as the k of two
// matrix steps.  Bound by the matrix instructions (16 of 64 cycles per KB of
// operands at T = 4).  The library's product does the whole matrix: 8000 rows
// of 8000 15.5 ms, here 9.3;
// 2583 of 1387 and the transpose 0.51 ms together, here 0.42; 500 of 500 20 us,
// here 15.
template <int T, int KS>
__global__ void __launch_bounds__(256, T == 4 ? 2 : 4) k_rdm_gram(int n, int M, unsigned total,
                                                                 const double *__restrict__ w,
                                                                 double *__restrict__ G) {
  constexpr int PD = T == 4 ? 2 : 4, D = PD - 1;
  // blocks of one XCD take neighbouring tiles (tile row by tile row)
  const unsigned per = (total + 7) / 8, id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || id >= total) return;
  const unsigned tile = id / KS;
  int bi = (int)((sqrt(8.0 * tile + 1.0) - 1.0) * 0.5);
  while ((unsigned)bi * (bi + 1) / 2 > tile) bi--;
  while ((unsigned)(bi + 1) * (bi + 2) / 2 <= tile) bi++;
  const int bj = (int)(tile - (unsigned)bi * (bi + 1) / 2);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, q = lane & 15, g = lane >> 4, half = wv >> 1;
  const int i0 = (2 * bi + (KS == 2 ? (int)(id & 1) : half)) * 16 * T, j0 = (2 * bj + (wv & 1)) * 16 * T;
  const bool mine = j0 <= i0 && i0 < n;
  if (KS == 1 && !mine) return;
  typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // rows of odd length: any element
  const double *pa[T], *pb[T];
#pragma unroll
  for (int f = 0; f < T; f++) {
    pa[f] = w + (size_t)min(i0 + 16 * f + q, n - 1) * M;
    pb[f] = w + (size_t)min(j0 + 16 * f + q, n - 1) * M;
  }
  d4 acc[T][T];
#pragma unroll
  for (int f = 0; f < T; f++)
#pragma unroll
    for (int j = 0; j < T; j++) acc[f][j] = d4{0.0, 0.0, 0.0, 0.0};
  struct Ops {
    d2u a[T], b[T];
  };
  auto mac = [&](const Ops &o) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int f = 0; f < T; f++)
#pragma unroll
        for (int j = 0; j < T; j++)
          acc[f][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(u ? o.a[f].y : o.a[f].x, u ? o.b[j].y : o.b[j].x,
                                                           acc[f][j], 0, 0, 0);
  };
  const int all = M / 8, first = KS == 2 && half ? all / 2 : 0;
  const int end = !mine ? 0 : KS == 2 && !half ? all / 2 : all;
  if (first < end) {
    auto fetch = [&](int s, Ops &o) {
      const int k = 8 * min(s, end - 1) + 2 * g;
#pragma unroll
      for (int f = 0; f < T; f++) {
        o.a[f] = *reinterpret_cast<const d2u *>(pa[f] + k);
        o.b[f] = *reinterpret_cast<const d2u *>(pb[f] + k);
      }
    };
    Ops o[PD];
#pragma unroll
    for (int p = 0; p < D; p++) fetch(first + p, o[p]);
    int s = first;
    for (; s + PD <= end; s += PD)
#pragma unroll
      for (int p = 0; p < PD; p++) {
        fetch(s + p + D, o[(p + D) % PD]);
        mac(o[p]);
        __builtin_amdgcn_sched_barrier(0);  // keep the stages' loads in this order
      }
#pragma unroll
    for (int p = 0; p < D; p++)
      if (s + p < end) mac(o[p]);
  }
  if (M % 8 && mine && (KS == 1 || half)) {  // the columns left over, zeros past them
    const int k = 8 * all + 2 * g;
    Ops o;
#pragma unroll
    for (int f = 0; f < T; f++) {
      o.a[f] = d2u{k < M ? pa[f][k] : 0.0, k + 1 < M ? pa[f][k + 1] : 0.0};
      o.b[f] = d2u{k < M ? pb[f][k] : 0.0, k + 1 < M ? pb[f][k + 1] : 0.0};
    }
    mac(o);
  }
  if constexpr (KS == 2) {
    __shared__ d4 other[2][T * T][64];
    if (half)
#pragma unroll
      for (int f = 0; f < T; f++)
#pragma unroll
        for (int j = 0; j < T; j++) other[wv & 1][f * T + j][lane] = acc[f][j];
    __syncthreads();
    if (half || !mine) return;
#pragma unroll
    for (int f = 0; f < T; f++)
#pragma unroll
      for (int j = 0; j < T; j++) acc[f][j] += other[wv & 1][f * T + j][lane];
  }
#pragma unroll
  for (int f = 0; f < T; f++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int i = i0 + 16 * f + 4 * r + g;
      if (i >= n) continue;
#pragma unroll
      for (int j = 0; j < T; j++) {
        const int c = j0 + 16 * j + q;
        if (c < n) G[(size_t)i * n + c] = acc[f][j][r];
      }
    }
}

// Tiles of 64 x 64 where they give every SIMD two waves, else of 32 x 32.
static void rdm_gram(Context &c, int n, int M, const double *w, double *G) {
  auto tiles = [&](int T) {
    const size_t b = cdiv(n, 32 * T);
    return b * (b + 1) / 2;
  };
  const bool wide = tiles(4) >= 2 * (size_t)c.n_cu;
  const size_t total = wide ? tiles(4) : 2 * tiles(2);
  if (total >= (1u << 28)) throw Error(3, "rdm: Gram matrix too large for one launch");
  const dim3 grid((unsigned)((total + 7) / 8 * 8));
  if (wide)
    hipLaunchKernelGGL((k_rdm_gram<4, 1>), grid, dim3(256), 0, c.stream, n, M, (unsigned)total, w, G);
  else
    hipLaunchKernelGGL((k_rdm_gram<2, 2>), grid, dim3(256), 0, c.stream, n, M, (unsigned)total, w, G);
  check_launch("k_rdm_gram");
}

// The same double pairs from the Gram matrix (its lower triangle) instead of a
// dot product per pair: out[e - e0] = sign * G[I, J]
__global__ void __launch_bounds__(256) k_rdm_double_gram(int n, uint64_t e0, uint64_t e1,
                                                         const uint64_t *__restrict__ d_off,
                                                         const uint32_t *__restrict__ d_ket,
                                                         const uint32_t *__restrict__ d_orb,
                                                         const uint64_t *__restrict__ str,
                                                         const double *__restrict__ G,
                                                         double *__restrict__ out) {
  const uint64_t e = e0 + (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (e >= e1) return;
  const int I = row_of(d_off, n, e);
  const size_t J = d_ket[e];
  const uint32_t o = d_orb[e];
  const int i = o & 255, j = (o >> 8) & 255, a = (o >> 16) & 255, b = (o >> 24) & 255;
  const uint64_t bra = str[I];
  double sg = parity1r(bra, i, a) * parity1r(bra, j, b);
  if (a > j || b < i) sg = -sg;
  out[e - e0] = sg * G[J < (size_t)I ? (size_t)I * n + J : J * n + I];
}

// Same-spin OneDiff scatter for the single pairs e0 <= e < e1 of one spin:
// the pair's dot product from T (pair e at (e - e0)) or, when T is null,
// with its sign from the Gram matrix G.
__global__ void k_rdm_single_scatter(int n, int L, int spin, uint64_t e0, uint64_t e1,
                                     const uint64_t *__restrict__ s_off,
                                     const uint64_t *__restrict__ s_ent,
                                     const uint64_t *__restrict__ str,
                                     const double *__restrict__ T, const double *__restrict__ G,
                                     double *__restrict__ one, double *__restrict__ two) {
  const uint64_t e = e0 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e1) return;
  const size_t L2 = (size_t)L * L, L4 = L2 * L2, L3 = L2 * L;
  const int I = row_of(s_off, n, e);
  const uint64_t ent = s_ent[e];
  const uint32_t pq = (uint32_t)((ent >> 32) & 0x7fffffffull);
  const int p = pq / L, q = pq % L;  // p = bra-only (cr), q = ket-only (an)
  double t0;
  if (T) {
    t0 = T[e - e0];
  } else {
    const size_t J = (uint32_t)(ent & 0xffffffffull);
    const double g = G[J < (size_t)I ? (size_t)I * n + J : J * n + I];
    t0 = (ent >> 63) ? -g : g;
  }
  atomicAdd(&one[spin * L2 + p + (size_t)L * q], t0);
  const size_t bs = (size_t)(3 * spin) * L4;  // same-spin block
  uint64_t occ = str[I];
  while (occ) {
    const int k = __ffsll((unsigned long long)occ) - 1;
    occ &= occ - 1;
    if (k == p) continue;  // the excited orbital's own terms cancel exactly
    atomicAdd(&two[bs + q + L * k + L2 * p + L3 * k], t0);
    atomicAdd(&two[bs + k + L * q + L2 * k + L3 * p], t0);
    atomicAdd(&two[bs + q + L * k + L2 * k + L3 * p], -t0);
    atomicAdd(&two[bs + k + L * q + L2 * p + L3 * k], -t0);
  }
}

// TwoDiff scatter for same-spin double pairs e0 <= e < e1 (block 0 alpha,
// 3 beta); T holds pair e at (e - e0).
__global__ void k_rdm_double_scatter(int L, int spin, uint64_t e0, uint64_t e1,
                                     const uint32_t *__restrict__ d_orb,
                                     const double *__restrict__ T, double *__restrict__ two) {
  const uint64_t e = e0 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= e1) return;
  const size_t L2 = (size_t)L * L, L4 = L2 * L2;
  const uint32_t o = d_orb[e];
  const size_t i = o & 255, j = (o >> 8) & 255, a = (o >> 16) & 255, b = (o >> 24) & 255;
  const double t = T[e - e0];
  const size_t bs = (size_t)(3 * spin) * L4;
  atomicAdd(&two[bs + a + L * b + L2 * (i + L * j)], t);
  atomicAdd(&two[bs + b + L * a + L2 * (j + L * i)], t);
  atomicAdd(&two[bs + a + L * b + L2 * (j + L * i)], -t);
  atomicAdd(&two[bs + b + L * a + L2 * (i + L * j)], -t);
}

// Two-spin term.  A block takes one work item: an alpha pair index pq (p >=
// q; T[qp][sr] = T[pq][rs] gives the rest) and a run of its alpha pairs
// (I, J, s_a).  Per alpha pair the rows x = s_a w[I,:] and y = w[J,:] are
// staged in LDS, each followed by a zero, and
//   T[pq][u v] += sum over the columns k of s_u s_v x[k + u] y[k + v]
// is a product of two matrices gathered from them, (orbitals x columns)
// times (columns x orbitals), on the FP64 matrix cores: a step of four
// columns is one 16x16x4 operand per tile of 16 orbitals, lane l holding
// orbital l % 16 of column l / 16 (SpinTables::rc_tab), read from LDS at the
// table's string with the table's sign.  A hole column's members are K - u
// and its element is -s_u s_v y[K - u] x[K - v].  The accumulators stay in
// registers over the item's alpha pairs.  The singles outside the columns
// (pb) are summed entry by entry, one pair bin per lane, into LDS.  The
// occupation numbers, T[pq][kk] = sum_i n_k(i) x[i] y[i], are taken once per
// item from the sum over its alpha pairs of x[i] y[i].  The item's row of T
// is collected in LDS and added to T with atomics.
// The columns hold several times more products than there are singles, at
// many times the rate: the entry-by-entry form (436k multiply-adds per alpha
// pair of a 8000-string set at 36 orbitals, two random 8-byte LDS reads
// each, and the alpha pairs of q > p as well) and the occupation sums of
// every single pair took 261 + 184 ms for 8000 x 8000 strings; this kernel
// takes 46 ms (2583 x 1387 at 29 orbitals: 10.3 -> 1.9 ms, 500 x 500 at 16:
// 1.16 -> 0.13 ms).  What bounds it there is the chain of an alpha pair
// (stage two rows, barrier, steps): with 130 KB staged one block of 8
// wavefronts fits in a CU; the matrix instructions alone would take 18 ms.
// Two wavefronts per SIMD (512 threads) leave 256 registers each for up to 9
// tiles of accumulators (twice, as the compiler pipelines them), the x y
// products and the gathers; with 4 tiles of orbitals a block takes two of
// them as rows (UT) and blockIdx.y says which.
constexpr int kMmThreads = 512;
constexpr int kMmWaves = kMmThreads / 64;
constexpr int kMmRho = 16;  // x y products per thread kept in registers (ROWS): nb <= 8192

__device__ __forceinline__ double signed_by(double v, uint32_t high) {
  return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, v) ^ ((uint64_t)high << 32));
}
// A row of w: staged in LDS with a zero behind it (LDS), or where it is, n
// values long (no member: string n, a zero).
template <bool LDS>
struct Row {
  const double *p;
  uint32_t n;
  __device__ __forceinline__ double at(uint32_t i) const { return LDS || i < n ? p[i] : 0.0; }
};
// the value of tile t's member in the row, with its sign (and `flip`)
template <bool LDS>
__device__ __forceinline__ double member(const Row<LDS> &row, uint64_t w, int t, uint32_t flip) {
  const uint32_t v = (uint32_t)(w >> (16 * t));
  return signed_by(row.at(v & 0x7fffu), ((v & 0x8000u) << 16) ^ flip);
}

// The steps s0 + wave, + waves, ... < s1 of columns over all tiles: two
// steps at a time, one's gathers under the other's matrix instructions, the
// table words of the next two in flight.
template <int NT, int UT, bool LDS>
__device__ __forceinline__ void rdm_steps_all(d4 (&acc)[UT][NT], const uint64_t *__restrict__ tab, int s0, int s1,
                                              int u0, Row<LDS> a_row, Row<LDS> b_row, uint32_t flip) {
  const int lane = threadIdx.x & 63;
  int s = s0 + (int)(threadIdx.x >> 6);
  if (s >= s1) return;
  auto word = [&](int q) { return tab[(size_t)64 * (q < s1 ? q : s) + lane]; };
  auto gather = [&](uint64_t w, double (&a)[UT], double (&b)[NT]) {
#pragma unroll
    for (int t = 0; t < UT; t++) a[t] = member(a_row, w, u0 + t, flip);
#pragma unroll
    for (int t = 0; t < NT; t++) b[t] = member(b_row, w, t, 0u);
  };
  auto mac = [&](const double (&a)[UT], const double (&b)[NT]) {
#pragma unroll
    for (int i = 0; i < UT; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
  };
  uint64_t w0 = word(s), w1 = word(s + kMmWaves);
  for (; s + kMmWaves < s1; s += 2 * kMmWaves) {
    double a0[UT], b0[NT], a1[UT], b1[NT];
    gather(w0, a0, b0);
    gather(w1, a1, b1);
    w0 = word(s + 2 * kMmWaves);
    w1 = word(s + 3 * kMmWaves);
    mac(a0, b0);
    mac(a1, b1);
  }
  if (s < s1) {
    double a0[UT], b0[NT];
    gather(w0, a0, b0);
    mac(a0, b0);
  }
}

// The same over one tile t: one matrix instruction per step, so four steps
// at a time into two accumulators (an instruction waits for the sum it adds
// to).
template <bool LDS>
__device__ __forceinline__ void rdm_steps_one(d4 &acc, const uint64_t *__restrict__ tab, int s0, int s1, int t,
                                              Row<LDS> a_row, Row<LDS> b_row, uint32_t flip) {
  const int lane = threadIdx.x & 63;
  int s = s0 + (int)(threadIdx.x >> 6);
  if (s >= s1) return;
  auto word = [&](int q) { return tab[(size_t)64 * (q < s1 ? q : s) + lane]; };
  d4 odd = {0.0, 0.0, 0.0, 0.0};
  uint64_t w[4];
#pragma unroll
  for (int q = 0; q < 4; q++) w[q] = word(s + q * kMmWaves);
  for (; s + 3 * kMmWaves < s1; s += 4 * kMmWaves) {
    double a[4], b[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      a[q] = member(a_row, w[q], t, flip);
      b[q] = member(b_row, w[q], t, 0u);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) w[q] = word(s + (4 + q) * kMmWaves);
#pragma unroll
    for (int q = 0; q < 4; q += 2) {
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q], b[q], acc, 0, 0, 0);
      odd = __builtin_amdgcn_mfma_f64_16x16x4f64(a[q + 1], b[q + 1], odd, 0, 0, 0);
    }
  }
#pragma unroll
  for (int q = 0; q < 3; q++)
    if (s + q * kMmWaves < s1)
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(member(a_row, w[q], t, flip), member(b_row, w[q], t, 0u), acc, 0, 0,
                                                 0);
  acc += odd;
}

struct RdmRanges {
  int4 r[24];
  int n;
};

// ROWS: the two rows in LDS and the x y sums in registers; otherwise (rows
// too long) both rows are read where they are and the sums are in LDS.
template <int NT, int UT, bool ROWS>
__global__ void __launch_bounds__(kMmThreads) k_rdm_mixed(int nb, int K, int L, const uint4 *__restrict__ items,
                                                          const uint64_t *__restrict__ a_ent, RdmRanges rg,
                                                          const uint64_t *__restrict__ tab, int nslice,
                                                          const uint32_t *__restrict__ pb,
                                                          const uint64_t *__restrict__ pb_off,
                                                          const uint32_t *__restrict__ pb_len,
                                                          const uint32_t *__restrict__ pb_perm,
                                                          const uint64_t *__restrict__ b_str,
                                                          const double *__restrict__ w, double *__restrict__ Tm) {
  extern __shared__ double lds[];
  double *trow = lds;             // [K]
  double *xs = lds + K;           // ROWS: x then a zero; else the x y sums
  double *ys = xs + nb + 1;       // ROWS: y then a zero
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63;
  const int u0 = UT < NT ? (int)blockIdx.y * UT : 0;
  const bool rest = u0 == 0;  // entries outside the columns and occupation numbers: once
  const uint4 it = items[blockIdx.x];
  for (int i = tid; i < K; i += kMmThreads) trow[i] = 0.0;
  if (!ROWS)
    for (int i = tid; i < nb; i += kMmThreads) xs[i] = 0.0;
  __syncthreads();
  d4 acc[UT][NT];
#pragma unroll
  for (int i = 0; i < UT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  double rho[ROWS ? kMmRho : 1];
#pragma unroll
  for (int k = 0; k < (ROWS ? kMmRho : 1); k++) rho[k] = 0.0;
  for (uint32_t e = it.y; e < it.z; e++) {
    const uint64_t ent = a_ent[e];
    const double *xg = w + (size_t)(uint32_t)(ent & 0xffffffffull) * nb;
    const double *yg = w + (size_t)((ent >> 32) & 0x7fffffffull) * nb;
    const uint32_t neg = (uint32_t)(ent >> 63) << 31;
    const Row<ROWS> x = {ROWS ? xs : xg, (uint32_t)nb}, y = {ROWS ? ys : yg, (uint32_t)nb};
    if (ROWS) {
      // half a row of each at a time, every load before the first store; the
      // first half is loaded before the barrier that ends the previous
      // pair's reads (nb < 8192: two halves of 8 values per thread)
      double vx[8], vy[8];
      auto load = [&](int i0) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const int i = i0 + k * kMmThreads;
          vx[k] = i < nb ? signed_by(xg[i], neg) : 0.0;
          vy[k] = i < nb ? yg[i] : 0.0;
        }
      };
      auto store = [&](int i0) {
#pragma unroll
        for (int k = 0; k < 8; k++) {
          const int i = i0 + k * kMmThreads;
          if (i <= nb) {
            xs[i] = vx[k];
            ys[i] = vy[k];
          }
        }
      };
      load(tid);
      __syncthreads();
      store(tid);
      if (nb >= 8 * kMmThreads) {
        load(tid + 8 * kMmThreads);
        store(tid + 8 * kMmThreads);
      }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < kMmRho; k++) {
        const int i = tid + k * kMmThreads;
        if (i < nb) rho[k] += xs[i] * ys[i];
      }
    } else {
      for (int i = tid; i < nb; i += kMmThreads) xs[i] += signed_by(xg[i], neg) * yg[i];
    }
    const uint32_t sx = ROWS ? 0u : neg;  // the alpha sign, where x is not staged with it
    for (int q = 0; q < rg.n; q++) {
      const int4 r = rg.r[q];
      const Row<ROWS> ar = r.w ? y : x, br = r.w ? x : y;
      const uint32_t flip = sx ^ (r.w ? 0x80000000u : 0u);
      if (r.z < 0) {
        rdm_steps_all<NT, UT, ROWS>(acc, tab, r.x, r.y, u0, ar, br, flip);
      } else if (r.z >= u0 && r.z < u0 + UT) {
        const int t = r.z;
        if (t == 0) rdm_steps_one<ROWS>(acc[0][0], tab, r.x, r.y, t, ar, br, flip);
        if constexpr (NT > 1)
          if (t == 1) rdm_steps_one<ROWS>(acc[1][1], tab, r.x, r.y, t, ar, br, flip);
        if constexpr (NT > 2)
          if (t == 2) rdm_steps_one<ROWS>(acc[UT == 2 ? 0 : 2][2], tab, r.x, r.y, t, ar, br, flip);
        if constexpr (NT > 3)
          if (t == 3) rdm_steps_one<ROWS>(acc[1][3], tab, r.x, r.y, t, ar, br, flip);
      }
    }
    if (rest)
      for (int sl = wv; sl < nslice; sl += kMmWaves) {
        const uint32_t len = pb_len[sl];
        const uint32_t *p = pb + pb_off[sl] + lane;
        double s = 0.0;
#pragma unroll 8
        for (uint32_t k = 0; k < len; k++) {
          const uint32_t wd = p[64 * (size_t)k];
          const uint32_t i = wd & 0x7fffu, j = (wd >> 15) & 0x7fffu;
          s += signed_by(x.at(i) * y.at(j), (wd & 0x80000000u) ^ sx);
        }
        const uint32_t bin = pb_perm[sl * 64 + lane];
        if (bin != 0xffffffffu) atomicAdd(&trow[bin], s);
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < UT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        // accumulator r of lane l: row 4 r + l / 16, column l % 16
        const int u = 16 * (u0 + i) + 4 * r + (lane >> 4), v = 16 * j + (lane & 15);
        if (u < L && v < L && u != v) atomicAdd(&trow[u * L + v], acc[i][j][r]);
      }
  if (rest) {  // the occupation numbers: lane = orbital, wavefront = a run of strings
    if (ROWS) {
#pragma unroll
      for (int k = 0; k < kMmRho; k++) {
        const int i = tid + k * kMmThreads;
        if (i < nb) xs[i] = rho[k];
      }
    }
    __syncthreads();
    const int per = (nb + kMmWaves - 1) / kMmWaves;
    const int i0 = wv * per, i1 = i0 + per < nb ? i0 + per : nb;
    double s = 0.0;
#pragma unroll 8
    for (int i = i0; i < i1; i++) s += ((b_str[i] >> lane) & 1ull) ? xs[i] : 0.0;
    if (lane < L) atomicAdd(&trow[lane * (L + 1)], s);
  }
  __syncthreads();
  for (int i = tid; i < K; i += kMmThreads) {
    const double v = trow[i];
    if (v != 0.0) atomicAdd(&Tm[(size_t)it.x * K + i], v);
  }
}

// Place T[pq][rs] (alpha p, q; beta r, s; rows p >= q are stored).  Two
// excitations (p != q and r != s) follow TwoDiffCorrelation's rules on the
// sorted spin orbitals I<J (bra-only 2p, 2r+1) and A<B (ket-only 2q, 2s+1);
// an excitation beside an occupation number, or two occupation numbers,
// OneDiff's and ZeroDiff's: (q, s, p, r) in the alpha-beta block, (s, q, r,
// p) in the beta-alpha block.
__global__ void k_rdm_mixed_place(int L, const double *__restrict__ Tm, double *__restrict__ two) {
  const size_t K = (size_t)L * L;
  const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= K * K) return;
  const int pq = (int)(idx / K), rs = (int)(idx % K);
  const int p = pq / L, q = pq % L, r = rs / L, s = rs % L;
  const double t = p >= q ? Tm[idx] : Tm[(size_t)(q * L + p) * K + s * L + r];
  if (t == 0.0) return;
  const size_t L2 = K, L4 = K * K;
  if (p == q || r == s) {
    atomicAdd(&two[2 * L4 + q + L * s + L2 * (p + L * r)], t);
    atomicAdd(&two[1 * L4 + s + L * q + L2 * (r + L * p)], t);
    return;
  }
  const int i = 2 * p, j = 2 * r + 1, a = 2 * q, b = 2 * s + 1;
  const int I = i < j ? i : j, J = i < j ? j : i, A = a < b ? a : b, B = a < b ? b : a;
  const size_t oi = I >> 1, si = I & 1, oa = A >> 1, sa = A & 1;
  const size_t oj = J >> 1, sj = J & 1, ob = B >> 1;
  // distinct (pq, rs) can land on one element, hence the atomics
  if (si == sa) {
    atomicAdd(&two[(si + 2 * sj) * L4 + oa + L * ob + L2 * (oi + L * oj)], t);
    atomicAdd(&two[(sj + 2 * si) * L4 + ob + L * oa + L2 * (oj + L * oi)], t);
  } else {
    atomicAdd(&two[(si + 2 * sj) * L4 + oa + L * ob + L2 * (oj + L * oi)], t);
    atomicAdd(&two[(sj + 2 * si) * L4 + ob + L * oa + L2 * (oi + L * oj)], t);
  }
}

template <int NT, int UT, bool ROWS>
static void launch_rdm_mixed(Context &c, const double *w, double *Tm) {
  auto fn = k_rdm_mixed<NT, UT, ROWS>;
  const size_t lds = sizeof(double) * ((size_t)c.K + (ROWS ? 2 * (c.nb + 1) : c.nb));
  SBDX_HIP(hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
  RdmRanges rg{};
  rg.n = c.B.rc_nrange;
  for (int i = 0; i < rg.n; i++) rg.r[i] = c.B.rc_range[i];
  if (c.A.ra_nitem == 0) return;
  hipLaunchKernelGGL(fn, dim3((unsigned)c.A.ra_nitem, NT / UT), dim3(kMmThreads), lds, c.stream, (int)c.nb, c.K, c.L,
                     (const uint4 *)c.A.ra_item, (const uint64_t *)c.A.ra_ent, rg, (const uint64_t *)c.B.rc_tab,
                     c.B.pb_nslice, (const uint32_t *)c.B.pb, (const uint64_t *)c.B.pb_off,
                     (const uint32_t *)c.B.pb_len, (const uint32_t *)c.B.pb_perm, (const uint64_t *)c.B.str, w, Tm);
  check_launch("k_rdm_mixed");
}
template <bool ROWS>
static void launch_rdm_mixed(Context &c, const double *w, double *Tm) {
  if (c.L <= 16) launch_rdm_mixed<1, 1, ROWS>(c, w, Tm);
  else if (c.L <= 32) launch_rdm_mixed<2, 2, ROWS>(c, w, Tm);
  else if (c.L <= 48) launch_rdm_mixed<3, 3, ROWS>(c, w, Tm);
  else launch_rdm_mixed<4, 2, ROWS>(c, w, Tm);
}

// p[0, n) = 0 (a fill kernel rather than hipMemsetAsync, so the work is a
// plain kernel sequence in every path)
__global__ void __launch_bounds__(256) k_rdm_zero(size_t n, double *__restrict__ p) {
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) p[i] = 0.0;
}

static void zero(Context &c, double *p, size_t n) {
  hipLaunchKernelGGL(k_rdm_zero, dim3((unsigned)std::min<size_t>(cdiv(n, 256), 4096)), dim3(256), 0, c.stream,
                     n, p);
  check_launch("k_rdm_zero");
}

// Working memory of one RDM evaluation: the mixed-term accumulator Tm[K][K]
// and room for td_cap double pairs; with G its Gram matrix, without it
// per-string sums and room for ts_cap single pairs (the pair tables are
// processed in chunks of that many entries).
struct RdmWork {
  double *rho_a, *rho_b, *Tm, *Ts, *Td;
  size_t ts_cap, td_cap;
  double *G = nullptr;  // room for max(na, nb)^2 values, or null (dot products per pair)
};

// Everything after the sign conversion: W' (alpha-first, device) to one and
// two (device, overwritten).  Kernels only, on c.stream; synchronizes once.
static void rdm_run(Context &c, const double *Wp, double *one, double *two, const RdmWork &wk) {
  const int L = c.L;
  const size_t L2 = (size_t)L * L, L4 = L2 * L2, K = (size_t)c.K;
  const int na = (int)c.na, nb = (int)c.nb;
  // beta sets up to 20000 strings and more, as far as one row and one row of
  // Tm fit in LDS (and 16-bit string numbers in the tables)
  const bool small = nb < 8192 && sizeof(double) * (2 * (size_t)nb + 2) <= c.lds_limit;
  if (nb >= 32767 || (!small && sizeof(double) * ((size_t)nb + K) > c.lds_limit))
    throw Error(3, "rdm: beta string count too large for the LDS-staged mixed RDM kernel");
  zero(c, one, 2 * L2);
  zero(c, two, 4 * L4);
  zero(c, wk.Tm, K * K);
  // W'^T (beta-major) for the beta-side sums
  transpose_into(c, Wp, c.T1, na, nb);
  // same-spin terms, alpha (rows of W') then beta (rows of W'^T), in chunks
  // of the pair tables
  for (int spin = 0; spin < 2; spin++) {
    const SpinTables &t = spin ? c.B : c.A;
    const double *w = spin ? c.T1 : Wp;
    const int M = spin ? na : nb;
    const bool gram = wk.G != nullptr;
    double *rho = spin ? wk.rho_b : wk.rho_a;
    if (gram) {
      rdm_gram(c, t.n, M, w, wk.G);
    } else {
      hipLaunchKernelGGL(k_rdm_diag_rows, dim3(t.n), dim3(256), 0, c.stream, M, w, rho);
      check_launch("k_rdm_diag_rows");
    }
    hipLaunchKernelGGL(k_rdm_diag_pairs, dim3(cdiv(t.n, 4 * kDiagStr)), dim3(256), sizeof(double) * L2, c.stream,
                       t.n, L, spin, t.str, gram ? (const double *)wk.G : (const double *)rho,
                       gram ? (size_t)t.n + 1 : 1, one, two);
    check_launch("k_rdm_diag_pairs");
    const size_t ts_cap = gram ? std::max<size_t>(t.ns, 1) : wk.ts_cap;
    for (size_t e0 = 0; e0 < t.ns; e0 += ts_cap) {
      const size_t e1 = std::min(t.ns, e0 + ts_cap);
      if (!gram) {
        hipLaunchKernelGGL(k_rdm_single_pairs, dim3((unsigned)std::min<size_t>(e1 - e0, 1u << 20)), dim3(256), 0,
                           c.stream, t.n, M, (uint64_t)e0, (uint64_t)e1, t.s_off, t.s_ent, w, wk.Ts);
        check_launch("k_rdm_single_pairs");
      }
      hipLaunchKernelGGL(k_rdm_single_scatter, dim3(cdiv(e1 - e0, 256)), dim3(256), 0, c.stream, t.n, L, spin,
                         (uint64_t)e0, (uint64_t)e1, t.s_off, t.s_ent, t.str, gram ? nullptr : wk.Ts, wk.G, one,
                         two);
      check_launch("k_rdm_single_scatter");
    }
    for (size_t e0 = 0; e0 < t.nd; e0 += wk.td_cap) {
      const size_t e1 = std::min(t.nd, e0 + wk.td_cap);
      if (gram) {
        hipLaunchKernelGGL(k_rdm_double_gram, dim3((unsigned)cdiv(e1 - e0, 256)), dim3(256), 0, c.stream, t.n,
                           (uint64_t)e0, (uint64_t)e1, t.d_off, t.d_ket, t.d_orb, t.str, wk.G, wk.Td);
        check_launch("k_rdm_double_gram");
      } else {
        hipLaunchKernelGGL(k_rdm_double_pairs, dim3((unsigned)std::min<size_t>(e1 - e0, 1u << 20)), dim3(256),
                           0, c.stream, t.n, M, (uint64_t)e0, (uint64_t)e1, t.d_off, t.d_ket, t.d_orb, t.str, w,
                           wk.Td);
        check_launch("k_rdm_double_pairs");
      }
      hipLaunchKernelGGL(k_rdm_double_scatter, dim3(cdiv(e1 - e0, 256)), dim3(256), 0, c.stream, L, spin,
                         (uint64_t)e0, (uint64_t)e1, t.d_orb, wk.Td, two);
      check_launch("k_rdm_double_scatter");
    }
  }
  // two spins: both rows staged when they fit beside the row of T (and the
  // x y sums in registers), else read where they are
  if (small && nb <= kMmRho * kMmThreads && sizeof(double) * (K + 2 * (size_t)nb + 2) <= c.lds_limit)
    launch_rdm_mixed<true>(c, Wp, wk.Tm);
  else
    launch_rdm_mixed<false>(c, Wp, wk.Tm);
  hipLaunchKernelGGL(k_rdm_mixed_place, dim3(cdiv(K * K, 256)), dim3(256), 0, c.stream, L, wk.Tm, two);
  check_launch("k_rdm_mixed_place");
  SBDX_HIP(hipStreamSynchronize(c.stream));
}

void compute_rdm(Context &c, const double *Wp, double *one, double *two) {
  ProfScope ps(c, "rdm");
  const size_t K = (size_t)c.K;
  const size_t ns = std::max<size_t>(std::max(c.A.ns, c.B.ns), 1);
  const size_t nd = std::max<size_t>(std::max(c.A.nd, c.B.nd), 1);
  TmpBuf b_tm(sizeof(double) * K * K), b_td(sizeof(double) * nd);
  RdmWork wk{nullptr, nullptr, (double *)b_tm.p, nullptr, (double *)b_td.p, ns, nd};
  // the Gram matrices of both spins' pairs when a quarter of free memory
  // holds one, else dot products per string and per pair
  const size_t mx = std::max(c.na, c.nb);
  size_t free_b = 0, total_b = 0;
  SBDX_HIP(hipMemGetInfo(&free_b, &total_b));
  std::unique_ptr<TmpBuf> b_g, b_rho, b_ts;
  if (mx < (1u << 31) && sizeof(double) * mx * mx < free_b / 4) {
    b_g.reset(new TmpBuf(sizeof(double) * mx * mx));
    wk.G = (double *)b_g->p;
  } else {
    b_rho.reset(new TmpBuf(sizeof(double) * (c.na + c.nb)));
    b_ts.reset(new TmpBuf(sizeof(double) * ns));
    wk.rho_a = (double *)b_rho->p;
    wk.rho_b = wk.rho_a + c.na;
    wk.Ts = (double *)b_ts->p;
  }
  rdm_run(c, Wp, one, two, wk);
}

// ---------------------------------------------------------------------------
// The same evaluation with working memory from a fixed static device array,
// for callers that cannot allocate (sbdx_rdm_device_noalloc).  Each device
// holds its own copy of `scratch` (kRdmScratchDoubles doubles = 128 MiB) from
// the first use of this file's kernels until the process ends.  In host code
// the array's name is only a stand-in: its device address comes from
// hipGetSymbolAddress, once per device, and only that address is passed on.
// Every call on one device shares the array, so calls that overlap on one
// device (other threads, other handles) race; the array keeps the last
// call's contents, and rdm_run clears what must start at zero.
constexpr size_t kRdmScratchDoubles = size_t(16) << 20;
static __device__ __align__(256) double scratch[kRdmScratchDoubles];

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[kMaxDevices] = {};

static double *scratch_address(int device) {
  if (device < 0 || device >= kMaxDevices) throw Error(3, "rdm (no-alloc): device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    SBDX_HIP(hipGetDevice(&cur));
    if (cur != device) throw Error(1, "rdm (no-alloc): call with the handle's device current");
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      throw Error(2, std::string("rdm (no-alloc): hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_ptr[device] = (double *)p;
  }
  return g_scratch_ptr[device];
}

// (na L of them are not used; they keep the largest instance that is
// accepted where it has always been)
size_t rdm_noalloc_fixed_doubles(const Context &c) {
  auto up = [](size_t n) { return (n + 31) & ~size_t(31); };  // 256-byte aligned regions
  return up(c.na) + up(c.nb) + up(c.na * (size_t)c.L) + up((size_t)c.K * c.K);
}

void compute_rdm_noalloc(Context &c, const double *Wp, double *one, double *two) {
  auto up = [](size_t n) { return (n + 31) & ~size_t(31); };
  const size_t L = (size_t)c.L, K = (size_t)c.K;
  const size_t fixed = rdm_noalloc_fixed_doubles(c);
  // at least 64 single pairs and 64 double pairs per chunk
  if (fixed + up(64 * (L + 1)) + up(64) > kRdmScratchDoubles) {
    char msg[256];
    snprintf(msg, sizeof msg,
             "rdm (no-alloc): the instance needs %zu + %zu doubles of working memory, more than the %zu "
             "(128 MiB) of the static scratch array",
             fixed, up(64 * (L + 1)) + up(64), kRdmScratchDoubles);
    throw Error(1, msg);
  }
  const int device = c.device;
  double *base = scratch_address(device);
  double *p = base;
  RdmWork wk{};
  wk.rho_a = p, p += up(c.na);
  wk.rho_b = p, p += up(c.nb);
  wk.Tm = p, p += up(K * K);
  const size_t rem = kRdmScratchDoubles - (size_t)(p - base);
  const size_t ns = std::max<size_t>(std::max(c.A.ns, c.B.ns), 1);
  const size_t nd = std::max<size_t>(std::max(c.A.nd, c.B.nd), 1);
  // half the rest for single pairs, the remainder for double pairs
  wk.ts_cap = std::min(ns, std::max<size_t>(64, rem / 2));
  wk.Ts = p, p += up(wk.ts_cap);
  wk.td_cap = std::min(nd, kRdmScratchDoubles - (size_t)(p - base));
  wk.Td = p;
  rdm_run(c, Wp, one, two, wk);
}

}  // namespace sbdx
