// The FP64 same-spin terms y = hii*x + H_a X + X H_b (X the na x nb vector)
// on the matrix cores.
//
// H_a and H_b hold the singles and doubles within one string set, some 10 to
// 25% of their elements.  Rows whose strings agree in their lowest orbitals
// (bit-reversed order: the same holes, then neighbouring particles) have most
// of their kets in common, so a tile of neighbouring rows meets only part of
// the set: of 8000 strings over 36 orbitals, 64 rows 57% of the kets (128
// rows 71%, 256 rows 90%; in the caller's order 64 rows meet all).  A tile
// keeps its kets as a list and the values over that list densely, in the
// order in which the matrix instructions take them; the product gathers x's
// rows by the list.  FP64 matrix instructions are slow enough (64 cycles
// each here) that operands come straight from memory into registers one
// stage ahead: no LDS, no barriers.
#include <algorithm>
#include <string>
#include <vector>

#include "common.h"

namespace sbdx {

namespace {

inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

typedef double d2 __attribute__((ext_vector_type(2)));
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));  // a pair at any element
typedef double d4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

constexpr int kStage = 8;  // kets a stage: two matrix steps of 4

// ---------------------------------------------------------------- tables
// One block per tile of tm rows: the kets of its rows as a bit set over the
// order (order[pos[r]] = r), counted (FILL false), or listed with the values (FILL true).
// List slot of ket k of a stage: 2 (k % 4) + k / 4 (a lane group takes its
// two kets with one load).  Value of row 16 f + m and ket k at
// [k / 4][f / 2][16 (k % 4) + m][f % 2] from base * tm on.
template <bool FILL>
__global__ void __launch_bounds__(256) k_tiles(int n, int tm, const uint32_t *__restrict__ rows,
                                               const uint32_t *__restrict__ order, const uint32_t *__restrict__ pos, const uint64_t *__restrict__ s_off,
                                               const uint64_t *__restrict__ s_ent, const double *__restrict__ s_val,
                                               const uint64_t *__restrict__ d_off, const uint32_t *__restrict__ d_ket,
                                               const double *__restrict__ d_val, uint32_t *__restrict__ cnt,
                                               const uint32_t *__restrict__ base, uint32_t *__restrict__ list,
                                               double *__restrict__ val) {
  extern __shared__ uint32_t bits[];
  __shared__ uint32_t sums[257];
  const int nw = (n + 31) / 32, tid = threadIdx.x, t = blockIdx.x;
  uint32_t *before = bits + nw;  // FILL: set bits of the words before each
  for (int i = tid; i < nw; i += 256) bits[i] = 0;
  __syncthreads();
  for (int m = 0; m < tm; m++) {
    const uint32_t r = rows[(size_t)t * tm + m];
    if (r >= (uint32_t)n) continue;
    for (uint64_t e = s_off[r] + tid; e < s_off[r + 1]; e += 256) {
      const uint32_t p = pos[s_ent[e] & 0xffffffffull];
      atomicOr(&bits[p >> 5], 1u << (p & 31));
    }
    for (uint64_t e = d_off[r] + tid; e < d_off[r + 1]; e += 256) {
      const uint32_t p = pos[d_ket[e]];
      atomicOr(&bits[p >> 5], 1u << (p & 31));
    }
  }
  __syncthreads();
  const int per = (nw + 255) / 256, w0 = min(nw, tid * per), w1 = min(nw, w0 + per);
  uint32_t s = 0;
  for (int i = w0; i < w1; i++) s += __popc(bits[i]);
  sums[tid + 1] = s;
  if (tid == 0) sums[0] = 0;
  __syncthreads();
  if (tid == 0)
    for (int i = 0; i < 256; i++) sums[i + 1] += sums[i];
  __syncthreads();
  if (!FILL) {
    if (tid == 0) cnt[t] = sums[256];
    return;
  }
  const size_t b0 = base[t], b1 = base[t + 1];
  uint32_t q = sums[tid];
  auto slot = [](uint32_t k) { return (k & ~7u) + 2 * (k & 3) + ((k >> 2) & 1); };
  for (int i = w0; i < w1; i++) {
    before[i] = q;
    for (uint32_t o = bits[i]; o; o &= o - 1, q++) {
      const uint32_t ket = order[32 * i + __ffs(o) - 1];
      list[b0 + slot(q)] = ket;
      if (q + 1 == sums[256])  // the last one again up to the stage's end, with zero values
        for (uint32_t k = q + 1; k < (uint32_t)(b1 - b0); k++) list[b0 + slot(k)] = ket;
    }
  }
  double *v = val + b0 * tm;
  for (size_t i = tid; i < (b1 - b0) * tm; i += 256) v[i] = 0.0;
  __syncthreads();
  auto put = [&](int m, uint32_t p, double x) {
    const uint32_t k = before[p >> 5] + __popc(bits[p >> 5] & ((1u << (p & 31)) - 1u));
    const int f = m >> 4;
    v[(size_t)(k >> 2) * 4 * tm + (f >> 1) * 128 + 2 * (16 * (k & 3) + (m & 15)) + (f & 1)] = x;
  };
  for (int m = 0; m < tm; m++) {
    const uint32_t r = rows[(size_t)t * tm + m];
    if (r >= (uint32_t)n) continue;
    for (uint64_t e = s_off[r] + tid; e < s_off[r + 1]; e += 256) put(m, pos[s_ent[e] & 0xffffffffull], s_val[e]);
    for (uint64_t e = d_off[r] + tid; e < d_off[r + 1]; e += 256) put(m, pos[d_ket[e]], d_val[e]);
  }
}

// ---------------------------------------------------------------- product
// y[r][c] = (DIAG ? hii x : 0) + sum_ket H[r][ket] x[ket][c], c < M.  A wave
// holds a tile of 16 MT rows by 16 NT columns (two columns of each pair of
// instructions adjacent: one 16-byte load); a block's four waves share the
// tile's values: side by side (KS 1), or two and two with half the list each
// (KS 2, sums added in LDS: at 32 x 32, where a wave or two per SIMD is all
// there is, twice as many shorter ones spread evenly).  Consecutive blocks of
// one XCD take the row tiles of one column chunk, walking their lists at the
// same pace, so x's rows come from that XCD's L2.
// Bound by the matrix instructions: 16 of them, 1024 cycles, per 8 KB of
// operands at 64 x 64.  One term of 8000 x 8000 strings 8.8 ms (7.4 at the
// instructions' rate over the tiles), as a dense library product 14.3; of 4001 x
// 4001 1.44 ms (1.09), as a dense library product 1.86; of 2583 x 2583 0.42 ms
// at 32 x 32 (with whole lists 0.46); both terms at 1000 x 900 0.10 ms with
// their transposes, in the small form below 0.19.  blockIdx.y: one of several
// vectors, vs elements from the one before.
template <int MT, int NT, int KS, bool DIAG>
__global__ void __launch_bounds__(256, MT == 4 ? 2 : 4)
    k_tile_mm(int n, int M, int ntile, int nchunk, const uint32_t *__restrict__ rows,
              const uint32_t *__restrict__ base, const uint32_t *__restrict__ list, const double *__restrict__ val,
              const double *__restrict__ x, const double *__restrict__ hii, double *__restrict__ y, size_t vs) {
  constexpr int TM = 16 * MT;
  x += blockIdx.y * vs;
  y += blockIdx.y * vs;
  const unsigned total = (unsigned)ntile * nchunk, per = (total + 7) / 8;
  const unsigned id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((blockIdx.x >> 3) >= per || id >= total) return;
  const int t = id % ntile, wv = threadIdx.x >> 6, lane = threadIdx.x & 63, g = lane >> 4;
  const int half = KS == 2 ? wv >> 1 : 0, side = KS == 2 ? wv & 1 : wv;
  const int c0 = ((int)(id / ntile) * (4 / KS) + side) * 16 * NT + 2 * (lane & 15);
  if (KS == 1 && c0 - 2 * (lane & 15) >= M) return;
  const double *xc[NT / 2];
#pragma unroll
  for (int j = 0; j < NT / 2; j++) xc[j] = x + min(c0 + 32 * j, M - 2);
  uint32_t b0 = base[t], nst = (base[t + 1] - b0) / kStage;
  if (KS == 2) {
    const uint32_t first = nst / 2;
    b0 += half ? first * kStage : 0;
    nst = half ? nst - first : first;
  }
  const uint2 *lp = reinterpret_cast<const uint2 *>(list + b0) + g;
  const d2 *vp = reinterpret_cast<const d2 *>(val + (size_t)b0 * TM) + lane;
  d4 acc[MT][NT];
#pragma unroll
  for (int f = 0; f < MT; f++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[f][j] = d4{0.0, 0.0, 0.0, 0.0};
  struct Ops {
    d2 a[2][MT / 2], b[2][NT / 2];
  };
  auto fetch = [&](uint32_t s, uint2 k, Ops &o) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const size_t row = (size_t)(u ? k.y : k.x) * M;
#pragma unroll
      for (int j = 0; j < NT / 2; j++) o.b[u][j] = *reinterpret_cast<const d2u *>(xc[j] + row);
#pragma unroll
      for (int f = 0; f < MT / 2; f++) o.a[u][f] = vp[(size_t)s * (kStage * TM / 2) + u * (2 * TM) + f * 64];
    }
  };
  auto mac = [&](const Ops &o) {
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int f = 0; f < MT; f++)
#pragma unroll
        for (int j = 0; j < NT; j++) acc[f][j] = mfma(o.a[u][f / 2][f & 1], o.b[u][j / 2][j & 1], acc[f][j]);
  };
  // PD stages in registers, PD - 1 of them on the way while one is worked on,
  // and the kets of as many more (stage t's in kk[t % PD])
  constexpr int PD = MT == 4 ? 2 : 4;
  if (nst) {
    const uint32_t last = nst - 1;
    auto kets = [&](uint32_t s) { return lp[4 * (size_t)min(s, last)]; };
    Ops o[PD];
    uint2 kk[PD];
#pragma unroll
    for (int p = 0; p < PD; p++) kk[(PD - 1 + p) % PD] = kets(PD - 1 + p);
#pragma unroll
    for (int p = 0; p < PD - 1; p++) fetch(min((uint32_t)p, last), kets(p), o[p]);
    constexpr int D = PD - 1;
    uint32_t s = 0;
    for (; s + PD <= nst; s += PD)
#pragma unroll
      for (int p = 0; p < PD; p++) {
        fetch(min(s + p + D, last), kk[(p + D) % PD], o[(p + D) % PD]);
        kk[(p + D) % PD] = kets(s + p + D + PD);
        mac(o[p]);
        __builtin_amdgcn_sched_barrier(0);  // keep the stages' loads in this order
      }
#pragma unroll
    for (int p = 0; p < D; p++)
      if (s + p < nst) mac(o[p]);
  }
  if constexpr (KS == 2) {
    __shared__ d4 other[2][MT * NT][64];
    if (half)
#pragma unroll
      for (int f = 0; f < MT; f++)
#pragma unroll
        for (int j = 0; j < NT; j++) other[side][f * NT + j][lane] = acc[f][j];
    __syncthreads();
    if (half) return;
#pragma unroll
    for (int f = 0; f < MT; f++)
#pragma unroll
      for (int j = 0; j < NT; j++) acc[f][j] += other[side][f * NT + j][lane];
  }
#pragma unroll
  for (int f = 0; f < MT; f++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const uint32_t row = rows[(size_t)t * TM + 16 * f + 4 * r + g];
      if (row >= (uint32_t)n) continue;
#pragma unroll
      for (int j = 0; j < NT / 2; j++) {
        const int c = c0 + 32 * j;
        const size_t at = (size_t)row * M + c;
        d2 v = {acc[f][2 * j][r], acc[f][2 * j + 1][r]};
        if (c + 1 < M) {
          if (DIAG) v += *reinterpret_cast<const d2u *>(hii + at) * *reinterpret_cast<const d2u *>(x + at);
          *reinterpret_cast<d2u *>(y + at) = v;
        } else if (c < M) {  // the last column of an odd row: the pair loaded was (M - 2, M - 1)
          y[at] = DIAG ? hii[at] * x[at] + v.y : v.y;
        }
      }
    }
}

// Small sets: one block per 16 x 16 tile of y, both terms in one pass over
// the dense blocks, the matrix steps of na + nb kets dealt to the four waves
// and their sums added at the end.  Bound by the reads of the operands (1 KB
// an instruction, no reuse between tiles), but one launch: 14 us at 300 x 280
// strings, where two library GEMMs after a pass for the diagonal took 45.
// blockIdx.z: one of several contiguous vectors.
__global__ void __launch_bounds__(256) k_same_small(int na, int nb, const double *__restrict__ Ha,
                                                    const double *__restrict__ Hb, const double *__restrict__ hii,
                                                    const double *__restrict__ x, double *__restrict__ y) {
  __shared__ double part[4][256];
  const int tid = threadIdx.x, wv = tid >> 6, lane = tid & 63, q = lane & 15, g = lane >> 4;
  const int r0 = blockIdx.y * 16, c0 = blockIdx.x * 16;
  x += (size_t)blockIdx.z * na * nb;
  y += (size_t)blockIdx.z * na * nb;
  const int rq = min(r0 + q, na - 1), cq = min(c0 + q, nb - 1);
  d4 acc = d4{0.0, 0.0, 0.0, 0.0}, odd = acc;
  // step s: kets 4 s + g of H_a x (s < sa), then of x H_b; past the end zeros
  const int sa = (na + 3) / 4, ns = sa + (nb + 3) / 4;
  auto fetch = [&](int s, double &a, double &b) {
    a = b = 0.0;
    if (s < sa) {
      const int k = 4 * s + g;
      if (k < na) a = Ha[(size_t)k * na + rq], b = x[(size_t)k * nb + cq];
    } else if (s < ns) {
      const int k = 4 * (s - sa) + g;
      if (k < nb) a = x[(size_t)rq * nb + k], b = Hb[(size_t)k * nb + cq];
    }
  };
  double a[4], b[4];
#pragma unroll
  for (int u = 0; u < 4; u++) fetch(wv + 4 * u, a[u], b[u]);
  for (int s = wv; s < ns; s += 16) {
    double an[4], bn[4];
#pragma unroll
    for (int u = 0; u < 4; u++) fetch(s + 16 + 4 * u, an[u], bn[u]);
    acc = mfma(a[0], b[0], acc);
    odd = mfma(a[1], b[1], odd);
    acc = mfma(a[2], b[2], acc);
    odd = mfma(a[3], b[3], odd);
#pragma unroll
    for (int u = 0; u < 4; u++) a[u] = an[u], b[u] = bn[u];
  }
#pragma unroll
  for (int r = 0; r < 4; r++) part[wv][(4 * r + g) * 16 + q] = acc[r] + odd[r];
  __syncthreads();
  const int r = r0 + (tid >> 4), c = c0 + (tid & 15);
  if (r >= na || c >= nb) return;
  const size_t at = (size_t)r * nb + c;
  y[at] = hii[at] * x[at] + ((part[0][tid] + part[1][tid]) + (part[2][tid] + part[3][tid]));
}

inline uint64_t bit_reverse(uint64_t v) {
  uint64_t r = 0;
  for (int i = 0; i < 64; i++) r |= ((v >> i) & 1ull) << (63 - i);
  return r;
}

// Small while one launch without reuse is no slower than four with it: 57 us
// against 61 at 600 x 590 strings, 79 against 77 at 700 x 700.
// A set of one string has no pair of columns to load.
bool small(const Context &c) { return c.na + c.nb <= kSameSmall || c.na == 1 || c.nb == 1; }

void build_tiles(Context &c, const SpinTables &t, const std::vector<uint64_t> &strs, size_t cols, SameTiles &o) {
  const int n = t.n;
  // 64 rows a tile where that gives every SIMD at least two waves of 64
  // columns, else 32 rows and 32 columns
  o.tm = (size_t)cdiv(n, 64) * cdiv(cols, 64) >= (size_t)8 * c.n_cu ? 64 : 32;
  o.ntile = (int)cdiv(n, o.tm);
  std::vector<uint64_t> rev(n);
  for (int i = 0; i < n; i++) rev[i] = bit_reverse(strs[i]);
  std::vector<uint32_t> order((size_t)o.ntile * o.tm, 0xffffffffu), pos(n);
  for (int i = 0; i < n; i++) order[i] = (uint32_t)i;
  std::stable_sort(order.begin(), order.begin() + n, [&](uint32_t a, uint32_t b) { return rev[a] < rev[b]; });
  for (int i = 0; i < n; i++) pos[order[i]] = (uint32_t)i;
  auto put = [&](const std::vector<uint32_t> &v) {
    uint32_t *p = (uint32_t *)dalloc(c, sizeof(uint32_t) * v.size());
    SBDX_HIP(hipMemcpyAsync(p, v.data(), sizeof(uint32_t) * v.size(), hipMemcpyHostToDevice, c.stream));
    return p;
  };
  std::vector<uint32_t> cnt(o.ntile), base(o.ntile + 1, 0), by(o.ntile), rows(order.size());
  TmpBuf tord(sizeof(uint32_t) * order.size()), tpos(sizeof(uint32_t) * n), tcnt(sizeof(uint32_t) * o.ntile);
  const StreamWait wait(c);
  SBDX_HIP(hipMemcpyAsync(tord.p, order.data(), sizeof(uint32_t) * order.size(), hipMemcpyHostToDevice, c.stream));
  SBDX_HIP(hipMemcpyAsync(tpos.p, pos.data(), sizeof(uint32_t) * n, hipMemcpyHostToDevice, c.stream));
  const uint32_t *dord = (const uint32_t *)tord.p, *dpos = (const uint32_t *)tpos.p;
  const size_t lds = sizeof(uint32_t) * 2 * ((n + 31) / 32);
  hipLaunchKernelGGL((k_tiles<false>), dim3((unsigned)o.ntile), dim3(256), lds, c.stream, n, o.tm, dord, dord, dpos,
                     t.s_off, t.s_ent, t.s_val, t.d_off, t.d_ket, t.d_val, (uint32_t *)tcnt.p,
                     (const uint32_t *)nullptr, (uint32_t *)nullptr, (double *)nullptr);
  check_launch("k_tiles");
  SBDX_HIP(hipMemcpyAsync(cnt.data(), tcnt.p, sizeof(uint32_t) * o.ntile, hipMemcpyDeviceToHost, c.stream));
  SBDX_HIP(hipStreamSynchronize(c.stream));
  // the tiles with the longest lists first (those of the reference string and
  // its singles meet all kets, twice the usual): a launch ends with short ones
  for (int i = 0; i < o.ntile; i++) by[i] = (uint32_t)i;
  std::stable_sort(by.begin(), by.end(), [&](uint32_t a, uint32_t b) { return cnt[a] > cnt[b]; });
  for (int i = 0; i < o.ntile; i++) {
    base[i + 1] = base[i] + (cnt[by[i]] + kStage - 1) / kStage * kStage;
    std::copy_n(order.begin() + (size_t)by[i] * o.tm, o.tm, rows.begin() + (size_t)i * o.tm);
  }
  o.rows = put(rows);
  o.base = put(base);
  o.list = (uint32_t *)dalloc(c, sizeof(uint32_t) * base[o.ntile]);
  o.val = (double *)dalloc(c, sizeof(double) * o.tm * (size_t)base[o.ntile]);
  hipLaunchKernelGGL((k_tiles<true>), dim3((unsigned)o.ntile), dim3(256), lds, c.stream, n, o.tm, o.rows, dord, dpos,
                     t.s_off, t.s_ent, t.s_val, t.d_off, t.d_ket, t.d_val, (uint32_t *)nullptr, o.base, o.list,
                     o.val);
  check_launch("k_tiles");
  SBDX_HIP(hipStreamSynchronize(c.stream));
}

// for k contiguous vectors
template <bool DIAG>
void tile_mm(Context &c, const SameTiles &o, int n, int M, const double *x, const double *hii, double *y, int k = 1) {
  const int nchunk = (int)cdiv(M, o.tm == 64 ? 256 : 64);
  if (M < 2 && n > 1) throw Error(3, "same-spin tiles: one column");
  const size_t blocks = (size_t)8 * cdiv((size_t)o.ntile * nchunk, 8);
  if (blocks >= (1ull << 31)) throw Error(3, "sigma: grid too large for one launch");
  if (o.tm == 64)
    hipLaunchKernelGGL((k_tile_mm<4, 4, 1, DIAG>), dim3((unsigned)blocks, k), dim3(256), 0, c.stream, n, M, o.ntile,
                       nchunk, o.rows, o.base, o.list, o.val, x, hii, y, (size_t)n * M);
  else
    hipLaunchKernelGGL((k_tile_mm<2, 2, 2, DIAG>), dim3((unsigned)blocks, k), dim3(256), 0, c.stream, n, M, o.ntile,
                       nchunk, o.rows, o.base, o.list, o.val, x, hii, y, (size_t)n * M);
  check_launch("k_tile_mm");
}

// The tiles, built on first use: all of their tables or none, so that a call
// after a failed one starts anew.
const SameTiles &tiles_of(Context &c, const SpinTables &t, const std::vector<uint64_t> &strs, size_t cols,
                          SameTiles &o) {
  if (o.val) return o;
  SameTiles n;
  try {
    build_tiles(c, t, strs, cols, n);
  } catch (...) {
    dfree(c, n.rows), dfree(c, n.base), dfree(c, n.list), dfree(c, n.val);
    throw;
  }
  return o = n;
}
const SameTiles &tiles_a(Context &c) { return tiles_of(c, c.A, c.h_astr, c.nb, c.tiles_a); }
const SameTiles &tiles_b(Context &c) {
  return c.B.alias ? tiles_a(c) : tiles_of(c, c.B, c.h_bstr, c.na, c.tiles_b);
}

}  // namespace

size_t same_mm_bytes(const Context &c) {
  auto one = [](size_t n) { return sizeof(double) * n * n; };
  return (c.tiles_a.val ? 0 : one(c.na)) + (c.B.alias || c.tiles_b.val ? 0 : one(c.nb));
}

// The tables take a bit set of the strings in LDS (a fourth of a byte per
// string, of 64 KB) and 32-bit offsets.
bool same_mm_fits(const Context &c) {
  auto one = [](size_t n) { return n <= (1u << 17) && (n + 63) / 32 * (n + 8) < (1ull << 32); };
  return one(c.na) && one(c.nb);
}

// Where the sets have few singles and doubles (random strings), the row
// kernels over them are faster than tiles that are nearly all zeros: at 60
// multiply-adds of the matrix cores per entry (the rates of the two forms,
// 70 and 1.3 TFLOP/s at 8000 x 8000 strings); and a single row or column of a
// large set would read its whole dense block.  Up to kSameSmall the one
// launch saves 9 us of launches and takes 0.092 us per 1e6 multiply-adds, the
// row kernels 1.4 us per 1e6 entries: a product of random strings over 40
// orbitals takes 32 us with the dense blocks and 38 with the rows at 250 x
// 250, 58 and 46 at 500 x 500, 85 and 60 at 600 x 600; over 24 orbitals 85
// and 80 at 600 x 600 (18e6 entries), 90 and 102 at 600 x 590 (33e6).
bool same_mm_worth(const Context &c) {
  const double work = (double)c.N * ((double)c.na + (double)c.nb);
  const double ent = (double)(c.A.ns + c.A.nd) * (double)c.nb + (double)(c.B.ns + c.B.nd) * (double)c.na;
  if (c.na + c.nb <= kSameSmall) return work <= 1e8 + 15.0 * ent;
  return !small(c) && work <= 60.0 * ent;
}

// y = hii*x + H_a X + X H_b for k contiguous vectors on the tiles; xt and yt:
// k N doubles each
static void tiles_both(Context &c, int k, const double *x, double *y, double *xt, double *yt) {
  const int na = (int)c.na, nb = (int)c.nb;
  tile_mm<true>(c, tiles_a(c), na, nb, x, c.hii, y, k);
  // the beta term with the vectors transposed, so that it gathers rows too
  transpose_into(c, x, xt, na, nb, k);
  tile_mm<false>(c, tiles_b(c), nb, na, xt, nullptr, yt, k);
  transpose_add(c, yt, y, nb, na, k);
}

static void small_both(Context &c, int k, const double *x, double *y) {
  const int na = (int)c.na, nb = (int)c.nb;
  double *Ha, *Hb;
  dense_blocks(c, Ha, Hb);
  hipLaunchKernelGGL(k_same_small, dim3(cdiv(nb, 16), cdiv(na, 16), k), dim3(256), 0, c.stream, na, nb,
                     (const double *)Ha, (const double *)Hb, c.hii, x, y);
  check_launch("k_same_small");
}

// y = hii*x + H_a X + X H_b; xt and yt: N doubles each
void same_mm(Context &c, const double *x, double *y, double *xt, double *yt) {
  if (small(c)) small_both(c, 1, x, y);
  else tiles_both(c, 1, x, y, xt, yt);
}

// The same for k contiguous vectors: a launch takes as many as kBlockDoubles
// hold, so that sets whose single vectors leave CUs idle fill the chip.  The
// one-launch form while its work is small: two vectors of 380 x 380 strings 31
// us against 38 on the tiles, four 50 and 50, two of 500 x 500 60 and 45.  One
// vector after the other, eight of 500 x 500 took 257 us, now 107; of 700 x
// 700 398 and 244 (batched library products 107 and 265).
void same_mm_block(Context &c, int k, const double *x, double *y, double *xt, double *yt) {
  constexpr size_t kBlockDoubles = size_t(4) << 20;
  const size_t N = c.N;
  const int group = (int)std::min<size_t>({(size_t)k, kBlockDoubles / N, 65535});
  const bool one = small(c) && (c.na == 1 || c.nb == 1 || (double)group * N * (c.na + c.nb) <= 4e8);
  if (group > 1 && !one && c.same_ws_cap < 2 * group * N) {
    try {
      double *p = (double *)dalloc(c, sizeof(double) * 2 * group * N);
      dfree(c, c.same_ws);
      c.same_ws = p;
      c.same_ws_cap = 2 * group * N;
    } catch (const Error &) {  // no room: one vector at a time
    }
  }
  for (int v = 0, n; v < k; v += n) {
    n = std::min(group, k - v);
    if (n > 1 && one) {
      small_both(c, n, x + v * N, y + v * N);
    } else if (n > 1 && c.same_ws_cap >= 2 * n * N) {
      tiles_both(c, n, x + v * N, y + v * N, c.same_ws, c.same_ws + n * N);
    } else {
      n = 1;
      same_mm(c, x + v * N, y + v * N, xt, yt);
    }
  }
}

// G = H_a X (a single string has an empty list)
void same_mm_alpha(Context &c, const double *x, double *G) {
  tile_mm<false>(c, tiles_a(c), (int)c.na, (int)c.nb, x, nullptr, G);
}

}  // namespace sbdx
