// Spin-orbital apply on a full particle-number set of sectors (FqeDataSet).
//
// The set holds every (nalpha, nbeta) sector with nalpha + nbeta = nele and
// both counts <= norb, in ascending nbeta, concatenated into one complex128
// vector of length L (each sector row-major lena x lenb).  Spin-orbital
// index p < norb is alpha orbital p, p >= norb beta orbital p - norb, and
// M = 2 norb.  For a target determinant I and an ordered pair (p, q) there
// is at most one source determinant J with <I|a+_p a_q|J> != 0; every
// kernel here is a gather over that J, so no kernel writes to a location
// another thread writes and no atomics are used.
//
// Signs follow the reference: within one spin (-1)^(occupied orbitals
// strictly between i and j) (src/fqe/fci_graph.py:204-244); across spins
// (-1)^nalpha(J) times the parities of the sector-to-sector maps, which
// count the occupied orbitals above the orbital
// (src/fqe/fqe_data_set.py:737-796, src/fqe/fci_graph_set.py:137-150).
//
// Two forms of the 1+2-body apply:
//
// Pair form (2 or more electrons; its buffers fit the workspace).  With
// A_qs = a_s a_q, q < s,
//   H C = sum_(p<r) A+_pr sum_(q<s) W[pr][qs] A_qs C,
// W the antisymmetrised V.  The one-body rest h'' = h1' + sum_t V[pt][tq] of
// the normal ordering goes into W as well, through
// a+_p a_q = sum_r a+_p a+_r a_r a_q / (nele - 1).  The intermediate states
// have nele - 2 electrons and there are M (M - 1) / 2 pairs for M^2, so the
// contraction is 8 (M (M - 1) / 2)^2 C(M, nele - 2) flops where the E_pq form
// below takes 8 M^4 C(M, nele): at M = 16 and 8 electrons 0.9 for 6.8 GFLOP.
// Above half filling the intermediate space grows past the target's; the
// workspace bounds it to about twice the target, still half of the flops.
//   k_set_pair_w    the real block form of W
//   k_set_pair_dvec D[qs][K] = <K|A_qs C>
//   k_set_gemm      Y = W D
//   k_set_pair_out  out[I] = sum_(p<r in I) <I|A+_pr|K> Y[pr][K]
// Signs: the operators act on determinants ordered alpha before beta, lowest
// first; that differs from the sector-to-sector convention above by
// (-1)^(nele - 1) per spin flip, so for even nele the sectors of odd nbeta
// change sign on the way in and out.
// M = 16, 8 electrons, all kernels of an apply: 71 us (contraction 31), 670 us in
// the E_pq form (51 workgroups gathering 385 us, contraction 196, D 88).
//
// E_pq form, and the 1-body apply:
//   k_set_dvec  D[pq][I] = sum_J <I|E_pq|J> C[J]   (one thread per I)
//   k_set_expand_v  the real block form [[Vr, -Vi], [Vi, Vr]] of V, with
//               the block form of the row h1' under it for the apply
//   k_set_gemm  Y = V D as one real FP64 matrix-core GEMM, k = 2 M^2 and
//               m = 2 M^2 (+ 2 rows that hold sum_pq h1'[pq] D[pq])
//   k_set_out   out[I]   = Y[h1' row][I] + sum_pq <I|E_pq|J> Y[pq][J]
//               for the 1+2-body apply, or
//               out[I]   = sum_pq h1[pq] <I|E_pq|J> C[J] for the 1-body one.  D and Y are planar per pair:
// row 2 pq holds the real parts, row 2 pq + 1 the imaginary parts, L
// doubles each, so the GEMM sees them as real 2 M^2 x L matrices.
#include "fqehip_common.h"

namespace fqehip {
namespace {

constexpr int kSetMaxNorb = 16;
constexpr int kSetMaxSec = kSetMaxNorb + 1;
constexpr int kSetBlock = 256;
constexpr int kSetPairChunk = 64;   // pairs per k_set_dvec block row
constexpr int kPairChunk = 8;       // pairs per k_set_pair_dvec block row
constexpr int kPairWaves = 8;       // waves that share a determinant's pairs

typedef double set_double4 __attribute__((ext_vector_type(4)));

struct SetDesc {
  int64_t total;                 // L
  int norb, nele, nsec, nbmin;   // sector s has nbeta = nbmin + s
  int64_t off[kSetMaxSec + 1];   // sector offsets, off[nsec] = L
  int32_t lenb[kSetMaxSec];
  int32_t binom[kSetMaxNorb + 1][kSetMaxNorb + 1];
};

__device__ __forceinline__ int popc(uint32_t x) { return __popc(x); }

// The binomials in LDS: every rank is a chain of lookups at indexes of its
// own per lane, which from the kernel arguments are cached global loads.
struct Binom {
  int32_t c[kSetMaxNorb + 1][kSetMaxNorb + 1];
};

__device__ __forceinline__ void load_binom(const SetDesc& d, Binom* t) {
  constexpr int kN = (kSetMaxNorb + 1) * (kSetMaxNorb + 1);
  for (int i = threadIdx.x; i < kN; i += blockDim.x)
    (&t->c[0][0])[i] = (&d.binom[0][0])[i];
  __syncthreads();
}

// Address of an nele-electron string in the reference's order (ascending
// occupation tuples in lexicographic order):
// C(n, k) - 1 - sum_t C(n - 1 - c_t, k + 1 - t), occupied c_1 < ... < c_k.
__device__ __forceinline__ int32_t lex_rank(uint32_t s, int n, int k,
                                            const Binom& b) {
  int32_t r = b.c[n][k] - 1;
  int t = 1;
  while (s) {
    int c = __ffs(s) - 1;
    s &= s - 1;
    r -= b.c[n - 1 - c][k + 1 - t];
    ++t;
  }
  return r;
}

// Inverse of lex_rank: the mirrored set has colex rank C(n,k) - 1 - r.
__device__ __forceinline__ uint32_t lex_unrank(int32_t r, int n, int k,
                                               const Binom& b) {
  int32_t rem = b.c[n][k] - 1 - r;
  uint32_t s = 0;
  int x = n - 1;
  for (int i = k; i >= 1; --i) {
    while (b.c[x][i] > rem) --x;   // stops at x = i - 1 at the latest
    s |= 1u << (n - 1 - x);
    rem -= b.c[x][i];
    --x;
  }
  return s;
}

__device__ __forceinline__ int bits_between32(uint32_t s, int i, int j) {
  int lo = i < j ? i : j, hi = i < j ? j : i;
  uint32_t mask = ((1u << hi) - 1u) & ~((2u << lo) - 1u);
  return popc(s & mask);
}

// Target determinant of sector `sec` with strings (a, b).  For pair (p, q)
// returns false when <I|E_pq|J> = 0 for every J; otherwise the flat index
// of J in the set vector and its sign.
__device__ __forceinline__ bool set_source(int p, int q, int sec, int na,
                                           int nb, uint32_t a, uint32_t b,
                                           const SetDesc& d, const Binom& bin,
                                           int64_t* jflat, double* sign) {
  const int n = d.norb;
  if (p < n && q < n) {            // alpha a+_i a_j, same sector
    const int i = p, j = q;
    if (!((a >> i) & 1u)) return false;
    if (i != j && ((a >> j) & 1u)) return false;
    const uint32_t src = (a ^ (1u << i)) | (1u << j);
    *sign = (bits_between32(a, i, j) & 1) ? -1.0 : 1.0;
    const int32_t ia = lex_rank(src, n, na, bin);
    const int64_t lenb = d.lenb[sec];
    *jflat = d.off[sec] + ia * lenb + lex_rank(b, n, nb, bin);
    return true;
  }
  if (p >= n && q >= n) {          // beta a+_i a_j, same sector
    const int i = p - n, j = q - n;
    if (!((b >> i) & 1u)) return false;
    if (i != j && ((b >> j) & 1u)) return false;
    const uint32_t src = (b ^ (1u << i)) | (1u << j);
    *sign = (bits_between32(b, i, j) & 1) ? -1.0 : 1.0;
    const int64_t lenb = d.lenb[sec];
    *jflat = d.off[sec] + lex_rank(a, n, na, bin) * lenb + lex_rank(src, n, nb, bin);
    return true;
  }
  if (p < n) {                     // a+_{i alpha} a_{j beta}: J in (na-1, nb+1)
    const int i = p, j = q - n;
    if (!((a >> i) & 1u) || ((b >> j) & 1u)) return false;
    const int ssec = sec + 1;
    if (ssec >= d.nsec) return false;
    const uint32_t sa = a ^ (1u << i), sb = b | (1u << j);
    const int par = (na - 1) + popc(a >> (i + 1)) + popc(b >> (j + 1));
    *sign = (par & 1) ? -1.0 : 1.0;
    const int64_t lenb = d.lenb[ssec];
    *jflat = d.off[ssec] + lex_rank(sa, n, na - 1, bin) * lenb +
             lex_rank(sb, n, nb + 1, bin);
    return true;
  }
  {                                // a+_{i beta} a_{j alpha}: J in (na+1, nb-1)
    const int i = p - n, j = q;
    if (!((b >> i) & 1u) || ((a >> j) & 1u)) return false;
    const int ssec = sec - 1;
    if (ssec < 0) return false;
    const uint32_t sa = a | (1u << j), sb = b ^ (1u << i);
    const int par = na + popc(a >> (j + 1)) + popc(b >> (i + 1));
    *sign = (par & 1) ? -1.0 : 1.0;
    const int64_t lenb = d.lenb[ssec];
    *jflat = d.off[ssec] + lex_rank(sa, n, na + 1, bin) * lenb +
             lex_rank(sb, n, nb - 1, bin);
    return true;
  }
}

// Sector, counts and strings of flat index g (g < L).
__device__ __forceinline__ void locate(int64_t g, const SetDesc& d,
                                       const Binom& bin, int* sec, int* na,
                                       int* nb, uint32_t* a, uint32_t* b) {
  int s = 0;
  while (s + 1 < d.nsec && g >= d.off[s + 1]) ++s;
  *sec = s;
  *nb = d.nbmin + s;
  *na = d.nele - *nb;
  const int64_t r = g - d.off[s];
  const int64_t lenb = d.lenb[s];
  *a = lex_unrank(static_cast<int32_t>(r / lenb), d.norb, *na, bin);
  *b = lex_unrank(static_cast<int32_t>(r % lenb), d.norb, *nb, bin);
}

// One thread per determinant and blockIdx.y-th chunk of kSetPairChunk
// pairs, so that the grid has enough blocks to fill the chip.
__global__ void __launch_bounds__(kSetBlock)
k_set_dvec(SetDesc d, int m2, const double2* __restrict__ c,
           double* __restrict__ dvec) {
  __shared__ Binom bin;
  load_binom(d, &bin);
  const int64_t g = static_cast<int64_t>(blockIdx.x) * kSetBlock + threadIdx.x;
  if (g >= d.total) return;
  int sec, na, nb;
  uint32_t a, b;
  locate(g, d, bin, &sec, &na, &nb, &a, &b);
  const int m = 2 * d.norb;
  const int pq0 = blockIdx.y * kSetPairChunk;
  const int pq1 = pq0 + kSetPairChunk < m2 ? pq0 + kSetPairChunk : m2;
  for (int pq = pq0; pq < pq1; ++pq) {
    int64_t j;
    double sg;
    double re = 0.0, im = 0.0;
    if (set_source(pq / m, pq % m, sec, na, nb, a, b, d, bin, &j, &sg)) {
      const double2 x = c[j];
      re = sg * x.x;
      im = sg * x.y;
    }
    dvec[static_cast<int64_t>(2 * pq) * d.total + g] = re;
    dvec[static_cast<int64_t>(2 * pq + 1) * d.total + g] = im;
  }
}

// a[(2 pq + u) * 2 m2 + 2 rs + w] = [[Vr, -Vi], [Vi, Vr]][u][w] of
// V[pq][rs] (complex128 [m2][m2]) for rows < 2 m2; rows 2 m2 and 2 m2 + 1
// (when rows = 2 m2 + 2) hold the same block form of the row h1[rs].  One
// thread per element of a.
__global__ void __launch_bounds__(kSetBlock)
k_set_expand_v(int m2, int rows, const double2* __restrict__ v,
               const double2* __restrict__ h1, double* __restrict__ a) {
  const int64_t n2 = 2LL * m2;
  const int64_t e = static_cast<int64_t>(blockIdx.x) * kSetBlock + threadIdx.x;
  if (e >= rows * n2) return;
  const int64_t row = e / n2, col = e % n2;
  const double2 h = row < n2 ? v[(row >> 1) * m2 + (col >> 1)] : h1[col >> 1];
  const int u = static_cast<int>(row & 1), w = static_cast<int>(col & 1);
  a[e] = (u == w) ? h.x : (u == 0 ? -h.y : h.y);
}

// y[m][ncol] = a[m][k] b[k][ncol], all real row-major FP64, on
// v_mfma_f64_16x16x4f64 (A operand: row lane%16, k lane/16; B operand:
// k lane/16, column lane%16; result item i: row lane/16 + 4 i, column
// lane%16, the layout k_gemm_f64 stores).  Out-of-range rows, columns and
// k are read as zero and not written.
//
// A wave owns 16 x 16 tiles of R row tiles by C column tiles, so each A value
// it loads feeds C MFMAs and each B value R; a block of 4 waves covers 16 R
// rows x 64 C columns and shares its rows of a through LDS.  k goes in chunks
// of KC: while one is multiplied the next one's A values (to the other LDS
// buffer) and B values (direct to registers) are in flight; with a single
// k step in flight, two waves per SIMD do not cover the latency of a load
// (240 x 240 x 8008: 42 us, now 31).
template <int R, int C, int KC>
__global__ void __launch_bounds__(kSetBlock, 2)
k_set_gemm(int m, int k, const double* __restrict__ a, int64_t ncol,
           const double* __restrict__ b, double* __restrict__ y) {
  constexpr int kA = R * 16 * KC / kSetBlock;      // A values per thread
  static_assert(kA * kSetBlock == R * 16 * KC, "even LDS fill");
  __shared__ double sa[2][R * 16][KC + 1];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int64_t col0 =
      (static_cast<int64_t>(blockIdx.x) * 4 + wave) * (16 * C);
  const int row0 = blockIdx.y * R * 16;
  const int kl = lane >> 4;
  const int li = lane & 15;
  set_double4 acc[R][C];
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int u = 0; u < C; ++u) acc[t][u] = set_double4{0, 0, 0, 0};
  auto load = [&](int kc0, double (&an)[kA], double (&bn)[KC / 4][C]) {
#pragma unroll
    for (int j = 0; j < kA; ++j) {
      const int e = threadIdx.x + j * kSetBlock;
      const int gr = row0 + e / KC, gc = kc0 + e % KC;
      an[j] = (gr < m && gc < k) ? a[static_cast<int64_t>(gr) * k + gc] : 0.0;
    }
#pragma unroll
    for (int st = 0; st < KC / 4; ++st) {
      const int kk = kc0 + 4 * st + kl;
#pragma unroll
      for (int u = 0; u < C; ++u) {
        const int64_t col = col0 + u * 16 + li;
        bn[st][u] = (kk < k && col < ncol) ? b[static_cast<int64_t>(kk) * ncol + col]
                                           : 0.0;
      }
    }
  };
  auto chunk = [&](int buf, const double (&an)[kA], const double (&bv)[KC / 4][C],
                   int next, double (&a2)[kA], double (&b2)[KC / 4][C]) {
#pragma unroll
    for (int j = 0; j < kA; ++j) {
      const int e = threadIdx.x + j * kSetBlock;
      sa[buf][e / KC][e % KC] = an[j];
    }
    // the other buffer's readers passed the previous chunk's barrier before
    // their reads, and this one after them
    __syncthreads();
    load(next, a2, b2);
#pragma unroll
    for (int st = 0; st < KC / 4; ++st)
#pragma unroll
      for (int t = 0; t < R; ++t) {
        const double av = sa[buf][t * 16 + li][4 * st + kl];
#pragma unroll
        for (int u = 0; u < C; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv[st][u], acc[t][u], 0, 0, 0);
      }
  };
  // every wave runs the same chunks, so all reach every barrier; a chunk past
  // k is zeros
  double a0[kA], a1[kA], b0[KC / 4][C], b1[KC / 4][C];
  load(0, a0, b0);
  for (int kc0 = 0; kc0 < k; kc0 += 2 * KC) {
    chunk(0, a0, b0, kc0 + KC, a1, b1);
    chunk(1, a1, b1, kc0 + 2 * KC, a0, b0);
  }
#pragma unroll
  for (int u = 0; u < C; ++u) {
    const int64_t col = col0 + u * 16 + li;
    if (col >= ncol) continue;
#pragma unroll
    for (int t = 0; t < R; ++t) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = row0 + t * 16 + kl + 4 * i;
        if (r < m) y[static_cast<int64_t>(r) * ncol + col] = acc[t][u][i];
      }
    }
  }
}

// Pairs q < s of M spin orbitals, row by row.
__device__ __forceinline__ void pair_of(int x, int m, int* q, int* s) {
  int r = 0;
  while (x >= m - 1 - r) {
    x -= m - 1 - r;
    ++r;
  }
  *q = r;
  *s = r + 1 + x;
}

// The dvec form of the tensors (reference src/fqe/fqe_data_set.py:194-197):
// V[pq][rs] = -h2[p][r][q][s] and h1'[p][s] = h1[p][s] + sum_k h2[p][k][k][s],
// h1 in place.  One thread per element of V; the first M^2 also of h1.
__global__ void __launch_bounds__(kSetBlock)
k_set_tensors(int m, const double2* __restrict__ h2, double2* __restrict__ h1,
              double2* __restrict__ v) {
  const int e = blockIdx.x * kSetBlock + threadIdx.x;
  const int m2 = m * m;
  if (e >= m2 * m2) return;
  const int s = e % m, r = e / m % m, q = e / m2 % m, p = e / m2 / m;
  const double2 x = h2[((p * m + r) * m + q) * m + s];
  v[e] = make_double2(-x.x, -x.y);
  if (e < m2) {
    const int i = e / m, j = e % m;
    double2 h = h1[e];
    for (int k = 0; k < m; ++k) {
      const double2 y = h2[((i * m + k) * m + k) * m + j];
      h.x += y.x;
      h.y += y.y;
    }
    h1[e] = h;
  }
}

// W[pr][qs] in the block form of k_set_expand_v, [2 np][2 np]: the four
// orderings of V[pq][rs] a+_p a+_r a_s a_q, and the one-body rest where the
// pairs share an orbital.  One thread per element of W; M terms at most.
__global__ void __launch_bounds__(kSetBlock)
k_set_pair_w(int m, int np, double inv, const double2* __restrict__ v,
             const double2* __restrict__ h1, double* __restrict__ w) {
  const int e = blockIdx.x * kSetBlock + threadIdx.x;
  if (e >= np * np) return;
  int p, r, q, s;
  pair_of(e / np, m, &p, &r);
  pair_of(e % np, m, &q, &s);
  const int m2 = m * m;
  auto at = [&](int i, int j, int k, int l) {
    return v[static_cast<int64_t>(i * m + j) * m2 + k * m + l];
  };
  const double2 v0 = at(p, q, r, s), v1 = at(r, q, p, s);
  const double2 v2 = at(p, s, r, q), v3 = at(r, s, p, q);
  double re = (v0.x - v1.x) + (v3.x - v2.x);
  double im = (v0.y - v1.y) + (v3.y - v2.y);
  auto one_body = [&](int i, int j, double f) {
    double2 h = h1[i * m + j];
#pragma unroll 8
    for (int t = 0; t < m; ++t) {
      const double2 x = at(i, t, t, j);
      h.x += x.x;
      h.y += x.y;
    }
    re += f * h.x;
    im += f * h.y;
  };
  if (r == s) one_body(p, q, inv);
  if (p == q) one_body(r, s, inv);
  if (p == s) one_body(r, q, -inv);
  if (r == q) one_body(p, s, -inv);
  const int64_t n2 = 2 * np;
  double* o = w + 2LL * (e / np) * n2 + 2 * (e % np);
  *reinterpret_cast<double2*>(o) = make_double2(re, -im);
  *reinterpret_cast<double2*>(o + n2) = make_double2(im, re);
}

// (-1)^(occupied below q and below s) for the orbitals of K, as the sign bit
// of the sum of two counts.
__device__ __forceinline__ int pair_parity(uint32_t k, int q, int s) {
  return (popc(k & ((1u << q) - 1u)) + popc(k & ((1u << s) - 1u))) & 1;
}

// Flat index in the set of the determinant with spin-orbital bits x, and
// whether its sector's sign is turned (even nele, odd nbeta).
__device__ __forceinline__ int64_t set_index(uint32_t x, const SetDesc& d,
                                             const Binom& bin, int* turned) {
  const uint32_t a = x & ((1u << d.norb) - 1u), b = x >> d.norb;
  const int nb = popc(b);
  const int sec = nb - d.nbmin;
  *turned = (nb & ~d.nele) & 1;
  return d.off[sec] +
         static_cast<int64_t>(lex_rank(a, d.norb, d.nele - nb, bin)) * d.lenb[sec] +
         lex_rank(b, d.norb, nb, bin);
}

// D[qs][K] for the determinants K of dk (two electrons fewer than d), planar
// rows 2 qs and 2 qs + 1.  One thread per K and blockIdx.y-th chunk of pairs.
__global__ void __launch_bounds__(kSetBlock)
k_set_pair_dvec(SetDesc d, SetDesc dk, int np, const double2* __restrict__ c,
                double* __restrict__ dvec) {
  __shared__ Binom bin;
  load_binom(d, &bin);
  const int64_t g = static_cast<int64_t>(blockIdx.x) * kSetBlock + threadIdx.x;
  if (g >= dk.total) return;
  int sec, na, nb;
  uint32_t a, b;
  locate(g, dk, bin, &sec, &na, &nb, &a, &b);
  const uint32_t k = a | b << d.norb;
  const int m = 2 * d.norb;
  const int x0 = blockIdx.y * kPairChunk;
  const int x1 = x0 + kPairChunk < np ? x0 + kPairChunk : np;
  int q, s;
  pair_of(x0, m, &q, &s);
  for (int x = x0; x < x1; ++x) {
    const uint32_t add = 1u << q | 1u << s;
    double re = 0.0, im = 0.0;
    if (!(k & add)) {
      int turned;
      const double2 v = c[set_index(k | add, d, bin, &turned)];
      const double sg = (pair_parity(k, q, s) ^ turned) ? -1.0 : 1.0;
      re = sg * v.x;
      im = sg * v.y;
    }
    dvec[static_cast<int64_t>(2 * x) * dk.total + g] = re;
    dvec[static_cast<int64_t>(2 * x + 1) * dk.total + g] = im;
    if (++s == m) {
      ++q;
      s = q + 1;
    }
  }
}

// out[I] = sum over the occupied pairs p < r of I.  A workgroup takes 64
// determinants; its waves take every kPairWaves-th pair each (51 workgroups
// of one thread per determinant leave most of the chip idle) and are summed
// in LDS in wave order.
__global__ void __launch_bounds__(64 * kPairWaves)
k_set_pair_out(SetDesc d, SetDesc dk, const double* __restrict__ y,
               double2* __restrict__ out) {
  __shared__ Binom bin;
  load_binom(d, &bin);
  __shared__ double2 part[kPairWaves][64];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t g = static_cast<int64_t>(blockIdx.x) * 64 + lane;
  const int m = 2 * d.norb;
  double re = 0.0, im = 0.0;
  int nb = 0;
  if (g < d.total) {
    int sec, na;
    uint32_t a, b;
    locate(g, d, bin, &sec, &na, &nb, &a, &b);
    const uint32_t det = a | b << d.norb;
    int at = 0;
    for (uint32_t up = det; up; up &= up - 1) {
      const int p = __ffs(up) - 1;
      for (uint32_t ur = up & (up - 1); ur; ur &= ur - 1, ++at) {
        if (at % kPairWaves != wave) continue;
        const int r = __ffs(ur) - 1;
        const uint32_t k = det ^ (1u << p | 1u << r);
        int unused;
        const int64_t j = set_index(k, dk, bin, &unused);
        const int x = p * (2 * m - p - 1) / 2 + (r - p - 1);
        const double sg = pair_parity(k, p, r) ? -1.0 : 1.0;
        re += sg * y[static_cast<int64_t>(2 * x) * dk.total + j];
        im += sg * y[static_cast<int64_t>(2 * x + 1) * dk.total + j];
      }
    }
  }
  part[wave][lane] = make_double2(re, im);
  __syncthreads();
  if (wave == 0 && g < d.total) {
    for (int w = 1; w < kPairWaves; ++w) {
      re += part[w][lane].x;
      im += part[w][lane].y;
    }
    const double sg = (nb & ~d.nele) & 1 ? -1.0 : 1.0;
    out[g] = make_double2(sg * re, sg * im);
  }
}

// kPlanarG: out[I] = Y[2 m2][I] + i Y[2 m2 + 1][I]
//                    + sum_pq <I|E_pq|J> (Y[2 pq][J] + i Y[2 pq + 1][J]);
// otherwise: out[I] = sum_pq hg[pq] <I|E_pq|J> C[J], C interleaved.
template <bool kPlanarG>
__global__ void __launch_bounds__(kSetBlock)
k_set_out(SetDesc d, int m2, const double2* __restrict__ hg,
          const double* __restrict__ gsrc, double2* __restrict__ out) {
  __shared__ Binom bin;
  load_binom(d, &bin);
  const int64_t g = static_cast<int64_t>(blockIdx.x) * kSetBlock + threadIdx.x;
  if (g >= d.total) return;
  int sec, na, nb;
  uint32_t a, b;
  locate(g, d, bin, &sec, &na, &nb, &a, &b);
  const int m = 2 * d.norb;
  double re = 0.0, im = 0.0;
  if (kPlanarG) {
    re = gsrc[static_cast<int64_t>(2 * m2) * d.total + g];
    im = gsrc[static_cast<int64_t>(2 * m2 + 1) * d.total + g];
  }
  for (int pq = 0; pq < m2; ++pq) {
    int64_t j;
    double sg;
    if (set_source(pq / m, pq % m, sec, na, nb, a, b, d, bin, &j, &sg)) {
      if (kPlanarG) {
        re += sg * gsrc[static_cast<int64_t>(2 * pq) * d.total + j];
        im += sg * gsrc[static_cast<int64_t>(2 * pq + 1) * d.total + j];
      } else {
        const double xr = gsrc[2 * j], xi = gsrc[2 * j + 1];
        const double hr = sg * hg[pq].x, hi = sg * hg[pq].y;
        re += hr * xr - hi * xi;
        im += hr * xi + hi * xr;
      }
    }
  }
  out[g] = make_double2(re, im);
}

int64_t host_binom(int n, int k) {
  if (k < 0 || n < 0 || k > n) return 0;
  int64_t r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}

int make_desc(int norb, int nele, SetDesc* d) {
  FQEHIP_CHECK_ARG(norb >= 1 && norb <= kSetMaxNorb,
                   "set apply: norb %d outside 1..%d", norb, kSetMaxNorb);
  FQEHIP_CHECK_ARG(nele >= 0 && nele <= 2 * norb,
                   "set apply: nele %d outside 0..%d", nele, 2 * norb);
  *d = SetDesc{};
  d->norb = norb;
  d->nele = nele;
  d->nbmin = nele > norb ? nele - norb : 0;
  const int nbmax = nele < norb ? nele : norb;
  d->nsec = nbmax - d->nbmin + 1;
  for (int n = 0; n <= kSetMaxNorb; ++n)
    for (int k = 0; k <= kSetMaxNorb; ++k)
      d->binom[n][k] = static_cast<int32_t>(host_binom(n, k));
  int64_t off = 0;
  for (int s = 0; s < d->nsec; ++s) {
    const int nb = d->nbmin + s, na = nele - nb;
    d->off[s] = off;
    d->lenb[s] = static_cast<int32_t>(host_binom(norb, nb));
    off += host_binom(norb, na) * host_binom(norb, nb);
  }
  d->off[d->nsec] = off;
  d->total = off;
  return FQEHIP_OK;
}

}  // namespace
}  // namespace fqehip

using namespace fqehip;

extern "C" int64_t fqehip_set_length(int norb, int nele) {
  SetDesc d;
  if (make_desc(norb, nele, &d) != FQEHIP_OK) return -1;
  return d.total;
}

// Workspace: D (2 m2 L doubles), Y ((2 m2 + 2) L doubles), then the real
// block form of V with the h1' row ((2 m2 + 2) 2 m2 doubles).  The pair form
// keeps its D, Y and W in the same space.
extern "C" int64_t fqehip_set_workspace_bytes(int norb, int nele) {
  SetDesc d;
  if (make_desc(norb, nele, &d) != FQEHIP_OK) return -1;
  const int64_t m2 = 4LL * norb * norb;
  return ((4 * m2 + 2) * d.total + (2 * m2 + 2) * 2 * m2) *
         static_cast<int64_t>(sizeof(double));
}

extern "C" int fqehip_set_dvec(int norb, int nele, const double* d_coeff,
                               double* d_dvec, void* stream) {
  clear_error();
  SetDesc d;
  if (int rc = make_desc(norb, nele, &d)) return rc;
  FQEHIP_CHECK_ARG(d_coeff != nullptr && d_dvec != nullptr,
                   "fqehip_set_dvec: null pointer");
  if (d.total == 0) return FQEHIP_OK;
  const int m2 = 4 * norb * norb;
  const dim3 grid(blocks_for(d.total, kSetBlock),
                  (m2 + kSetPairChunk - 1) / kSetPairChunk);
  k_set_dvec<<<grid, kSetBlock, 0, as_stream(stream)>>>(d, m2,
                                    reinterpret_cast<const double2*>(d_coeff),
                                    d_dvec);
  FQEHIP_CHECK_LAUNCH("k_set_dvec");
  return FQEHIP_OK;
}

namespace fqehip {
namespace {

// y[m][ncol] = a[m][k] b[k][ncol].  64 x 256 tiles if they fill the chip
// twice over; else 32 x 128, four times as many.  Smaller / larger tiles, us:
// 240 x 240 x 8008 (128 large tiles) 32 / 49, 306 x 306 x 18564 (365) 99 / 102,
// 306 x 306 x 43758 (855) 221 / 206, 380 x 380 x 125970 (2958) 1031 / 873.
int set_gemm(int m, int k, const double* a, int64_t ncol, const double* b, double* y,
             hipStream_t st) {
  const int64_t large = static_cast<int64_t>(blocks_for(ncol, 256)) * ((m + 63) / 64);
  if (large >= 512)
    k_set_gemm<4, 4, 8><<<dim3(blocks_for(ncol, 256), (m + 63) / 64), kSetBlock, 0, st>>>(
        m, k, a, ncol, b, y);
  else
    k_set_gemm<2, 2, 32><<<dim3(blocks_for(ncol, 128), (m + 31) / 32), kSetBlock, 0, st>>>(
        m, k, a, ncol, b, y);
  FQEHIP_CHECK_LAUNCH("k_set_gemm");
  return FQEHIP_OK;
}

// Y = [V; h1'] D on the workspace (h1 may be null: V rows only).
int set_contract(const SetDesc& d, int m2, const double* v, const double* h1,
                 double* ws, hipStream_t st) {
  const int n2 = 2 * m2;
  const int rows = n2 + (h1 != nullptr ? 2 : 0);
  double* dv = ws;
  double* y = dv + static_cast<int64_t>(n2) * d.total;
  double* a = y + static_cast<int64_t>(n2 + 2) * d.total;
  const int64_t na = static_cast<int64_t>(rows) * n2;
  k_set_expand_v<<<blocks_for(na, kSetBlock), kSetBlock, 0, st>>>(
      m2, rows, reinterpret_cast<const double2*>(v),
      reinterpret_cast<const double2*>(h1), a);
  FQEHIP_CHECK_LAUNCH("k_set_expand_v");
  return set_gemm(rows, n2, a, d.total, dv, y, st);
}

// The pair form: whether it applies, and the apply.
bool pair_form(const SetDesc& d, SetDesc* dk, int64_t workspace) {
  if (d.nele < 2 || make_desc(d.norb, d.nele - 2, dk) != FQEHIP_OK) return false;
  const int64_t np = static_cast<int64_t>(d.norb) * (2 * d.norb - 1);
  return (4 * np * dk->total + 4 * np * np) * 8 <= workspace;
}

int pair_apply(const SetDesc& d, const SetDesc& dk, const double* h1, const double* v,
               const double2* c, double2* out, double* ws, hipStream_t st) {
  const int m = 2 * d.norb, np = m * (m - 1) / 2;
  double* dv = ws;
  double* y = dv + 2LL * np * dk.total;
  double* w = y + 2LL * np * dk.total;
  k_set_pair_w<<<blocks_for(static_cast<int64_t>(np) * np, kSetBlock), kSetBlock, 0, st>>>(
      m, np, 1.0 / (d.nele - 1), reinterpret_cast<const double2*>(v),
      reinterpret_cast<const double2*>(h1), w);
  FQEHIP_CHECK_LAUNCH("k_set_pair_w");
  k_set_pair_dvec<<<dim3(blocks_for(dk.total, kSetBlock), (np + kPairChunk - 1) / kPairChunk),
                    kSetBlock, 0, st>>>(d, dk, np, c, dv);
  FQEHIP_CHECK_LAUNCH("k_set_pair_dvec");
  if (int rc = set_gemm(2 * np, 2 * np, w, dk.total, dv, y, st)) return rc;
  k_set_pair_out<<<blocks_for(d.total, 64), 64 * kPairWaves, 0, st>>>(d, dk, y, out);
  FQEHIP_CHECK_LAUNCH("k_set_pair_out");
  return FQEHIP_OK;
}

}  // namespace
}  // namespace fqehip

extern "C" int fqehip_set_contract(int norb, int nele, const double* d_v,
                                   double* d_workspace, void* stream) {
  clear_error();
  SetDesc d;
  if (int rc = make_desc(norb, nele, &d)) return rc;
  FQEHIP_CHECK_ARG(d_v != nullptr && d_workspace != nullptr,
                   "fqehip_set_contract: null pointer");
  if (d.total == 0) return FQEHIP_OK;
  return set_contract(d, 4 * norb * norb, d_v, nullptr, d_workspace,
                      as_stream(stream));
}

extern "C" int fqehip_set_tensors(int norb, double* d_h1, const double* d_h2,
                                  double* d_v, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(norb >= 1 && norb <= kSetMaxNorb,
                   "set tensors: norb %d outside 1..%d", norb, kSetMaxNorb);
  FQEHIP_CHECK_ARG(d_h1 && d_h2 && d_v && d_v != d_h2,
                   "fqehip_set_tensors: null pointer or aliased output");
  const int m = 2 * norb;
  const int64_t n = static_cast<int64_t>(m) * m * m * m;
  k_set_tensors<<<blocks_for(n, kSetBlock), kSetBlock, 0, as_stream(stream)>>>(
      m, reinterpret_cast<const double2*>(d_h2), reinterpret_cast<double2*>(d_h1),
      reinterpret_cast<double2*>(d_v));
  FQEHIP_CHECK_LAUNCH("k_set_tensors");
  return FQEHIP_OK;
}

extern "C" int fqehip_set_apply(int norb, int nele, const double* d_h1,
                                const double* d_v, const double* d_coeff,
                                double* d_out, double* d_workspace,
                                void* stream) {
  clear_error();
  SetDesc d;
  if (int rc = make_desc(norb, nele, &d)) return rc;
  FQEHIP_CHECK_ARG(d_h1 != nullptr && d_coeff != nullptr && d_out != nullptr,
                   "fqehip_set_apply: null pointer");
  FQEHIP_CHECK_ARG(d_v == nullptr || d_workspace != nullptr,
                   "fqehip_set_apply: the two-body apply needs a workspace");
  FQEHIP_CHECK_ARG(d_coeff != d_out,
                   "fqehip_set_apply: output must not alias the input");
  if (d.total == 0) return FQEHIP_OK;
  const int m2 = 4 * norb * norb;
  const unsigned nblk = blocks_for(d.total, kSetBlock);
  hipStream_t s = as_stream(stream);
  const double2* h1 = reinterpret_cast<const double2*>(d_h1);
  const double2* c = reinterpret_cast<const double2*>(d_coeff);
  double2* out = reinterpret_cast<double2*>(d_out);
  if (d_v == nullptr) {
    k_set_out<false><<<nblk, kSetBlock, 0, s>>>(d, m2, h1, d_coeff, out);
    FQEHIP_CHECK_LAUNCH("k_set_out");
    return FQEHIP_OK;
  }
  SetDesc dk;
  if (pair_form(d, &dk, fqehip_set_workspace_bytes(norb, nele)))
    return pair_apply(d, dk, d_h1, d_v, c, out, d_workspace, s);
  double* dv = d_workspace;
  double* y = dv + 2LL * m2 * d.total;
  const dim3 dgrid(nblk, (m2 + kSetPairChunk - 1) / kSetPairChunk);
  k_set_dvec<<<dgrid, kSetBlock, 0, s>>>(d, m2, c, dv);
  FQEHIP_CHECK_LAUNCH("k_set_dvec");
  if (int rc = set_contract(d, m2, d_v, d_h1, d_workspace, s)) return rc;
  k_set_out<true><<<nblk, kSetBlock, 0, s>>>(d, m2, nullptr, y, out);
  FQEHIP_CHECK_LAUNCH("k_set_out");
  return FQEHIP_OK;
}
