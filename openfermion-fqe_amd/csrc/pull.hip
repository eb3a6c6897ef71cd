// Pull form of the complex128 two-body apply, without a dvec and without
// slot rows.
//
// Alpha and beta pair operators commute, so for any operator in the dvec
// form H = sum_pq V[p][q] E_p E_q + sum_q h1'[q] E_q, E_p = E^a_p + E^b_p
// (reference src/fqe/fqe_data.py:646-683), or with separate spin-orbital
// blocks (:712-741),
//
//   H C = Haa C + C Hbb^T + sum_q E^b_q ( sum_p W[p][q] E^a_p C ),
//
// Haa and Hbb the matrices of the operator on the strings of one spin
// (fqehip_spin_block), W[p][q] = V[p][q] + V[q][p] (alpha pair p, beta pair
// q) the opposite-spin coupling; the reference's lm kernels make the same
// three-way split (src/fqe/lib/fqe_data.c:668-720, :879-996).
//
//   k_same_spin_f64:  rowacc = Haa C + C Hbb^T, both products accumulated in
//       the same registers (one pass over K = lena, then over K = lenb);
//   k_pull_rows_f64:  one workgroup per alpha string ia.  E^a_p C at row ia
//       is +-C[src_p(ia), :], a whole row of C, so the contraction over p is
//       a GEMM of W (beta pairs x the live alpha pairs of ia) with rows of
//       C as they lie in memory, and E^b_q moves its result within row ia,
//       which is an accumulator row in LDS.
//
// Against the split form (beta excitations gathered, alpha excitations
// scattered to slot rows in HBM): the B operand needs no gather within the
// row, no sign and no conversion; K is the live alpha pairs (50 of 105 at
// norb 14) instead of all pairs; and the slot rows, nalpha (norb - nalpha)
// values of 16 bytes per determinant written and read again, are gone.  The
// price is the dense Haa C.
#include <type_traits>

#include "fqehip_common.h"
#include "pull_common.h"
#include "rows_common.h"

namespace fqehip {
namespace {

using namespace rows;

typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr size_t kLdsLimit = 160 * 1024;
constexpr int64_t kOffLimit = int64_t(1) << 31;   // 32-bit buffer offsets

__device__ __forceinline__ double u2d(uint32_t lo, uint32_t hi) {
  return __longlong_as_double(static_cast<long long>(
      static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32)));
}

// v with its sign flipped where bit 31 of sg is set
__device__ __forceinline__ double with_sign(double v, uint32_t sg) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
  return u2d(static_cast<uint32_t>(b), static_cast<uint32_t>(b >> 32) ^ sg);
}

// auxiliary bits of a buffer load: volatile (the compiler does not move it)
constexpr int kVolatile = static_cast<int>(0x80000000u);

// ---------------------------------------------------------------------------
// rowacc = Haa C + C Hbb^T
// ---------------------------------------------------------------------------
// Both products accumulate in the same registers: P[ia][k] Q[k][ib] over
// k < lena with P = Haa, Q = C, then over k < lenb with P = C, Q = Hbb.  A
// wave owns 16 RA x 16 RB complex outputs, a workgroup of 4 waves (2 x 2)
// the neighbouring ones.
//
// No LDS: every operand is loaded in the layout of v_mfma_f64_16x16x4f64
// (A: row l%16, k l/16; B: k l/16, column l%16) straight from memory, D k
// steps ahead in a register ring.  Haa, Hbb (stored by source string) and C
// as Q are runs of 16 consecutive elements per k; C as P is 64 bytes of 16
// rows, the other half of the cache line serving the next k step.  An MFMA
// takes 64 clocks, so a k step of 2 x 2 tiles (8 MFMAs, 512 clocks) needs 3 KB
// per wave, 24 bytes per clock and CU of the L1's 64 (2 x 4 tiles: 20), and
// the waves need no barrier and no staging work.  norb 14 7a7b (3.2e11
// flops): 4.7 ms, 69 TFLOP/s of the 78 that the instruction reaches, with 2 x 4
// tiles; 5.7 ms with 2 x 2; 5.7 ms with both operands staged through
// double-buffered LDS tiles of 64 x 64 (6.6 ms with 128 x 64).
//
// k past lena or lenb is out of range, hence zero, for H (and masked for C);
// columns past a row read what follows into outputs that are not stored.
constexpr int kSpinDepth = 4;              // k steps in flight

__device__ __forceinline__ double load_d(__amdgpu_buffer_rsrc_t r, int off) {
  const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
  return u2d(v[0], v[1]);
}

//
// SPLIT, for sectors whose tiles would leave most of the chip idle: the
// workgroup owns the outputs of one wave and each wave takes a quarter of
// both sums; the quarters are added in wave order (red: 4 x 256 RA RB values of
// LDS).  It shortens the chain of k steps by four and brings four times as
// many waves: 252 x 252 strings 20.6 -> 8.7 us, 330 x 462 30.8 -> 21.4.
template <bool CPLX, int RA, int RB, bool SPLIT>
__device__ __forceinline__ void same_spin_tile(
    int t, int64_t lena, int64_t lenb, const double* __restrict__ ha,
    const double* __restrict__ hb, const double* __restrict__ coeff,
    double* __restrict__ out, int ta, int tb, double2* red) {
  constexpr int D = SPLIT ? 2 * kSpinDepth : kSpinDepth;
  constexpr int kH = CPLX ? 16 : 8;               // bytes per H element
  // groups of 8 tile rows, so neighbouring workgroups share C and H rows
  const int grp = t / (8 * tb);
  const int left = ta - grp * 8;
  const int rows = left < 8 ? left : 8;
  const int w = t - grp * 8 * tb;
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int kq = lane >> 4;
  const int cl = lane & 15;
  const int ti = grp * 8 + w % rows, tj = w / rows;
  const int a0 = (SPLIT ? ti : ti * 2 + (wave >> 1)) * 16 * RA;
  const int b0 = (SPLIT ? tj : tj * 2 + (wave & 1)) * 16 * RB;
  const int la = static_cast<int>(lena), lb = static_cast<int>(lenb);
  if (a0 >= la || b0 >= lb) return;
  const __amdgpu_buffer_rsrc_t rc = buffer_of(coeff, lena * lenb * 16);
  const __amdgpu_buffer_rsrc_t rha = buffer_of(ha, lena * lena * kH);
  const __amdgpu_buffer_rsrc_t rhb = buffer_of(hb, lenb * lenb * kH);

  double4_t are[RA][RB], aim[RA][RB];
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j) {
      are[i][j] = double4_t{0, 0, 0, 0};
      aim[i][j] = double4_t{0, 0, 0, 0};
    }
  // the k steps of this wave: whole rings, so only the last ones can pass the end
  auto first = [&](int ns) { return SPLIT ? wave * ((ns + 4 * D - 1) / (4 * D)) * D : 0; };
  auto last = [&](int ns) {
    const int e = SPLIT ? (wave + 1) * ((ns + 4 * D - 1) / (4 * D)) * D : ns;
    return e < ns ? e : ns;
  };
  // an operand value of a k step: real and imaginary part (H: real only
  // unless CPLX)
  auto load_h = [&](__amdgpu_buffer_rsrc_t r, int off, double& re, double& im) {
    if constexpr (CPLX) {
      const double2 v = bload_d2(r, off);
      re = v.x;
      im = v.y;
    } else {
      re = load_d(r, off);
    }
  };
  {
    double pr[D][RA], pi[D][RA];
    double2 q[D][RB];
    auto load = [&](int s, int d) {
      const int k = 4 * s + kq;
#pragma unroll
      for (int i = 0; i < RA; ++i)
        load_h(rha, (k * la + a0 + 16 * i + cl) * kH, pr[d][i], pi[d][i]);
#pragma unroll
      for (int j = 0; j < RB; ++j)
        q[d][j] = bload_d2(rc, (k * lb + b0 + 16 * j + cl) * 16);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(first((la + 3) / 4) + d, d);
    const int end = last((la + 3) / 4);
    for (int s0 = first((la + 3) / 4); s0 < end; s0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int i = 0; i < RA; ++i)
#pragma unroll
          for (int j = 0; j < RB; ++j) {
            are[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[d][i], q[d][j].x, are[i][j], 0, 0, 0);
            aim[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(pr[d][i], q[d][j].y, aim[i][j], 0, 0, 0);
            if constexpr (CPLX) {
              are[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-pi[d][i], q[d][j].y, are[i][j], 0, 0, 0);
              aim[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(pi[d][i], q[d][j].x, aim[i][j], 0, 0, 0);
            }
          }
        load(s0 + d + D, d);
      }
    }
  }
  {
    double2 p[D][RA];
    double qr[D][RB], qi[D][RB];
    auto load = [&](int s, int d) {
      const int k = 4 * s + kq;
#pragma unroll
      for (int i = 0; i < RA; ++i)
        p[d][i] = bload_d2(rc, k < lb ? ((a0 + 16 * i + cl) * lb + k) * 16 : -1);
#pragma unroll
      for (int j = 0; j < RB; ++j)
        load_h(rhb, (k * lb + b0 + 16 * j + cl) * kH, qr[d][j], qi[d][j]);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) load(first((lb + 3) / 4) + d, d);
    const int end = last((lb + 3) / 4);
    for (int s0 = first((lb + 3) / 4); s0 < end; s0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
#pragma unroll
        for (int i = 0; i < RA; ++i)
#pragma unroll
          for (int j = 0; j < RB; ++j) {
            are[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(p[d][i].x, qr[d][j], are[i][j], 0, 0, 0);
            aim[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(p[d][i].y, qr[d][j], aim[i][j], 0, 0, 0);
            if constexpr (CPLX) {
              are[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-p[d][i].y, qi[d][j], are[i][j], 0, 0, 0);
              aim[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(p[d][i].x, qi[d][j], aim[i][j], 0, 0, 0);
            }
          }
        load(s0 + d + D, d);
      }
    }
  }
  // item e of lane l: row l/16 + 4 e, column l%16
  if constexpr (SPLIT) {
    constexpr int kOut = 256 * RA * RB;
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
      for (int j = 0; j < RB; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          red[wave * kOut + ((i * RB + j) * 4 + e) * 64 + lane] =
              make_double2(are[i][j][e], aim[i][j][e]);
    __syncthreads();
    // item (i, j, e) by wave e
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
      for (int j = 0; j < RB; ++j) {
        const double2* r = red + ((i * RB + j) * 4 + wave) * 64 + lane;
        double2 v = r[0];
#pragma unroll
        for (int q = 1; q < 4; ++q) {
          v.x += r[q * kOut].x;
          v.y += r[q * kOut].y;
        }
        const int a = a0 + 16 * i + kq + 4 * wave;
        const int b = b0 + 16 * j + cl;
        if (a < la && b < lb)
          *reinterpret_cast<double2*>(out + (static_cast<int64_t>(a) * lb + b) * 2) = v;
      }
    return;
  }
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int a = a0 + 16 * i + kq + 4 * e;
        const int b = b0 + 16 * j + cl;
        if (a < la && b < lb)
          *reinterpret_cast<double2*>(out + (static_cast<int64_t>(a) * lb + b) * 2) =
              make_double2(are[i][j][e], aim[i][j][e]);
      }
}

template <bool CPLX, int RA, int RB, bool SPLIT>
__global__ void __launch_bounds__(256, RA * RB > 4 || CPLX ? 2 : 4)
k_same_spin_f64(int64_t lena, int64_t lenb, const double* __restrict__ ha,
                const double* __restrict__ hb, const double* __restrict__ coeff,
                double* __restrict__ out, const int32_t* done, PullSeries series,
                int ta, int tb) {
  __shared__ double2 red[SPLIT ? 4 * 256 * RA * RB : 1];
  if (done && *done) return;
  if (series.partials && series_done(series, static_cast<int>(lena))) return;
  same_spin_tile<CPLX, RA, RB, SPLIT>(static_cast<int>(xcd_order(blockIdx.x, ta * tb)),
                                      lena, lenb, ha, hb, coeff, out, ta, tb, red);
}

template <bool CPLX, int RA, int RB, bool SPLIT = false>
void same_spin(int64_t lena, int64_t lenb, const double* ha, const double* hb,
               const double* coeff, double* out, const PullSeries& series,
               hipStream_t st, const int32_t* done) {
  constexpr int kRows = (SPLIT ? 16 : 32) * RA, kCols = (SPLIT ? 16 : 32) * RB;
  const int ta = static_cast<int>((lena + kRows - 1) / kRows);
  const int tb = static_cast<int>((lenb + kCols - 1) / kCols);
  k_same_spin_f64<CPLX, RA, RB, SPLIT><<<static_cast<unsigned>(ta * tb), 256, 0, st>>>(
      lena, lenb, ha, hb, coeff, out, done, series, ta, tb);
}

// ---------------------------------------------------------------------------
// Opposite-spin rows
// ---------------------------------------------------------------------------
constexpr int kPullMaxK = 64;              // live alpha pairs + folded row
constexpr int kPullTiles = 7;              // 16-row W tiles per pass
constexpr int kPullDepth = 4;              // k steps of B in flight
constexpr int kPullRows = kPullMaxK + 4 * kPullDepth;   // lrow entries
constexpr uint32_t kPullNoRow = 0x80000000u;   // past the end of C

constexpr int64_t kInRowMax = 5000;      // see pull_in_row

// The first beta pair of pass ps of G W tiles.  Passes are equal, so 9 tiles run
// as 2 x 5; the last pass begins early enough to end with the table of target
// words (the bounds check of its loads does not cover the row part of their
// address), with zeros for the rows of W that an earlier pass had.
__host__ __device__ __forceinline__ int pull_pass_start(int ps, int G, int nq) {
  const int last = 16 * ((nq + 15) / 16 - G);
  return 16 * G * ps < last ? 16 * G * ps : last;
}

struct PullArgs {
  int norb, compressed, nele, nq;          // nq: pairs of one spin
  int64_t lena, lenb;
  int ks, pass, copies;                    // k steps, passes, accumulator rows
  const double* w;                         // [p][q] (complex: interleaved)
  const int32_t* dexc;                     // [lena][nexc][3]
  const uint32_t* fwd;                     // fqehip_pull_table
  const double* coeff;
  double* rowacc;
  // out != NULL: out = alpha (rowacc + row) + beta cin, acc += that value;
  // else rowacc += row
  double alpha_re, alpha_im, beta_re, beta_im;
  const double* cin;
  double* out;
  double* acc;
  const double* acc0;                      // not NULL: acc = acc0 + that value
  double* partials;                        // not NULL: [ia] = |out row|^2
  const double* ha;                        // not NULL: the same-spin part is
  const double* hb;                        // computed here, not read
  PullSeries series;
  const int32_t* done;
};

size_t pull_lds_bytes(bool cplx, int ks, int64_t lenb, int tiles, int copies) {
  return static_cast<size_t>(copies) * lenb * 16 +
         static_cast<size_t>(tiles) * ks * 64 * 8 * (cplx ? 2 : 1) +
         kPullMaxK * (8 + 4 + 4) + kPullRows * 4 + 8 * 4;
}

// Row ia of Haa C + C Hbb^T into accumulator row 0.  Eight lanes share a
// column, each with every eighth term of both sums: the loads of a wave are
// 128-byte pieces of eight rows of C and 64-byte pieces of eight rows of Hbb.
// 32 terms of both make a step, and the next step's loads are in flight while
// one is summed (latency bounds it: with the rows, 70 x 70 strings take 13.4 us,
// 14.7 without the overlap, and 8 + 5.5 us as two kernels).
template <bool CPLX>
__device__ __forceinline__ void same_spin_row(const PullArgs& p, int64_t ia, int wave,
                                              int nwave, int lane, double2* accs) {
  constexpr int kH = CPLX ? 16 : 8;
  const int lena = static_cast<int>(p.lena), lenb = static_cast<int>(p.lenb);
  const int kp = lane & 7, xl = lane >> 3;
  const __amdgpu_buffer_rsrc_t rc = buffer_of(p.coeff, p.lena * p.lenb * 16);
  const __amdgpu_buffer_rsrc_t ra = buffer_of(p.ha, p.lena * p.lena * kH);
  const __amdgpu_buffer_rsrc_t rb = buffer_of(p.hb, p.lenb * p.lenb * kH);
  const int row = static_cast<int>(ia);
  const int nj = ((lena > lenb ? lena : lenb) + 31) / 32;
  struct Step {
    double2 h[8], c[8];
  };
  auto load_h = [&](__amdgpu_buffer_rsrc_t r, int off) {
    return CPLX ? bload_d2(r, off) : make_double2(load_d(r, off), 0.0);
  };
  // terms and columns past the last read zero
  auto load = [&](Step& s, int x0, int jb) {
    const int x = x0 + xl;
    const bool ok = x < lenb;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = 32 * jb + 8 * u + kp;
      const bool a = ok && j < lena, b = ok && j < lenb;
      s.h[u] = load_h(ra, a ? (j * lena + row) * kH : -1);
      s.c[u] = bload_d2(rc, a ? (j * lenb + x) * 16 : -1);
      s.h[4 + u] = load_h(rb, b ? (j * lenb + x) * kH : -1);
      s.c[4 + u] = bload_d2(rc, b ? (row * lenb + j) * 16 : -1);
    }
  };
  double re = 0.0, im = 0.0;
  int x0 = wave * 8, jb = 0;               // the step that is summed
  auto sum = [&](const Step& s) {
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      re += s.h[u].x * s.c[u].x;
      im += s.h[u].x * s.c[u].y;
      if (CPLX) {
        re -= s.h[u].y * s.c[u].y;
        im += s.h[u].y * s.c[u].x;
      }
    }
    if (++jb < nj) return;
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
      re += __shfl_xor(re, o);
      im += __shfl_xor(im, o);
    }
    if (kp == 0 && x0 + xl < lenb) accs[x0 + xl] = make_double2(re, im);
    re = im = 0.0;
    jb = 0;
    x0 += nwave * 8;
  };
  int lx = x0, lj = 0;                     // the next step to load
  auto next = [&](Step& s) {
    load(s, lx, lj);
    if (++lj == nj) {
      lj = 0;
      lx += nwave * 8;
    }
  };
  Step s0, s1;
  next(s0);
  while (x0 < lenb) {
    next(s1);
    sum(s0);
    if (x0 >= lenb) break;
    next(s0);
    sum(s1);
  }
}

// One alpha string ia per workgroup; G 16-row tiles of W per pass.
//
// Set-up: the live alpha pairs of ia are its de-excitation rows to another
// string (noff = nele (norb - nele) of them: source row of C, pair, sign),
// plus one folded row, C[ia] itself, whose coefficient is the sum over the
// occupied orbitals' diagonal pairs.  W restricted to them, with the signs,
// goes to LDS in MFMA A-operand order ([k step][tile][lane]).
//
// Then each wave takes 16-column tiles of the row in turn: the B operand of
// lane l (k = 4 s + l/16, column l%16) is the 16-byte value C[src_k][col], so
// the loads are the operand, kPullDepth steps ahead in a ring; each k step
// feeds G x (re, im) independent MFMAs; and the G x 16 values Z[q][col] are
// added, with the sign of E^b_q, to the accumulator row at their target
// column (ds_add_f64, about 10 clocks per wave instruction).
//
// Order of the additions: `copies` accumulator rows, wave w adding to row
// w % copies.  The waves that share one add in turn, tile after tile (`turn`,
// a counter per row in LDS: the tile whose turn it is), so every accumulator
// sees the same sequence of additions on every run, and the rows are summed
// in order at the end.  A wave waits only for waves with earlier tiles, and
// those for none after them, so every wait ends.
//
// norb 14 7a7b: 5.4 ms (2.7e11 flops with the padding, 50 TFLOP/s of 78), against
// 7.6 + 1.6 ms of the slot-row kernel and its reduction; 4.8 ms without the
// additions, 5.1 without their order.  norb 12 6a6b: 0.24 against 0.47 + 0.09;
// complex operator, norb 11 4a6b: 0.14 against 1.23 for the unfused kernels.
//
// Small sectors (pull_in_row) have no same-spin kernel before this one: see
// same_spin_row.
template <bool CPLX, int G>
__device__ __forceinline__ void pull_row(const PullArgs& p, int64_t ia,
                                         char* smem) {
  constexpr int kF = CPLX ? 128 : 64;      // doubles per W fragment
  const int tid = threadIdx.x;
  const int nt = blockDim.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nwave = nt >> 6;
  const int lane = tid & 63;
  const int kq = lane >> 4;
  const int cl = lane & 15;
  const int lenb = static_cast<int>(p.lenb);
  const int ks = p.ks;
  double2* accs = reinterpret_cast<double2*>(smem);    // [copies][lenb]
  double* wf = reinterpret_cast<double*>(accs + p.copies * lenb);   // [ks][G][kF]
  double* lsg = wf + G * ks * kF;
  uint32_t* lrow = reinterpret_cast<uint32_t*>(lsg + kPullMaxK);
  int32_t* lp = reinterpret_cast<int32_t*>(lrow + kPullRows);
  int32_t* ldiag = lp + kPullMaxK;
  int32_t* turns = ldiag + kPullMaxK;              // [8]
  const int noff = p.nele * (p.norb - p.nele);
  const int mine = wave % p.copies;
  // the table's offsets are those of element target + 1
  char* accum = reinterpret_cast<char*>(accs + mine * lenb) - 16;
  int32_t* turn = turns + mine;

  for (int x = tid; x < p.copies * lenb; x += nt) accs[x] = make_double2(0.0, 0.0);
  if (wave == 0) {
    const int nexc = p.nele * (p.norb - p.nele + 1);
    int32_t src = -1, ij = 0, sg = 0;
    if (lane < nexc) {
      const int32_t* e = p.dexc + (ia * nexc + lane) * 3;
      src = e[0];
      ij = e[1];
      sg = e[2];
    }
    const bool diag = lane < nexc && src == ia;
    const bool off = lane < nexc && src != ia;
    const uint64_t mo = __ballot(off), md = __ballot(diag);
    const uint64_t below = (1ull << lane) - 1ull;
    const int i = ij / p.norb, j = ij % p.norb;
    const int pair = p.compressed ? comp_pair(i, j) : ij;
    if (off) {
      const int pos = __popcll(mo & below);
      lrow[pos] = static_cast<uint32_t>(src) * static_cast<uint32_t>(lenb) * 16u;
      lp[pos] = pair;
      lsg[pos] = static_cast<double>(sg);
    }
    if (diag) ldiag[__popcll(md & below)] = pair;
    if (lane >= noff)
      lrow[lane] = lane == noff
                       ? static_cast<uint32_t>(ia) * static_cast<uint32_t>(lenb) * 16u
                       : kPullNoRow;
    if (lane < kPullRows - kPullMaxK) lrow[kPullMaxK + lane] = kPullNoRow;
  }
  __syncthreads();

  const __amdgpu_buffer_rsrc_t rc = buffer_of(p.coeff, p.lena * p.lenb * 16);
  const __amdgpu_buffer_rsrc_t rf = buffer_of(p.fwd, static_cast<int64_t>((p.nq + 15) & ~15) * lenb * 4);
  const __amdgpu_buffer_rsrc_t rw =
      buffer_of(p.w, static_cast<int64_t>(p.nq) * p.nq * (CPLX ? 16 : 8));
  const int ntile = (lenb + 15) >> 4;

  // ahead of the first addition: the barriers below are in between
  if (p.ha) same_spin_row<CPLX>(p, ia, wave, nwave, lane, accs);

  for (int ps = 0; ps < p.pass; ++ps) {
    const int q0 = pull_pass_start(ps, G, p.nq);
    const int qnew = 16 * G * ps;          // pairs before it: an earlier pass
    // elements of rows past the live ones, of pairs past the last or of an
    // earlier pass and of the folded row (next loop) are out of range and read
    // zero
#pragma unroll 4
    for (int f = wave; f < G * ks; f += nwave) {
      const int q = q0 + 16 * (f % G) + cl;
      const int k = 4 * (f / G) + kq;
      const int off = k < noff && q >= qnew && q < p.nq ? (lp[k] * p.nq + q) * (CPLX ? 16 : 8) : -1;
      const double sg = k < noff ? lsg[k] : 0.0;
      if (CPLX) {
        const double2 v = bload_d2(rw, off);
        wf[f * kF + lane] = sg * v.x;
        wf[f * kF + 64 + lane] = sg * v.y;
      } else {
        wf[f * kF + lane] = sg * load_d(rw, off);
      }
    }
    __syncthreads();
    for (int t = wave; t < G; t += nwave) {
      const int q = q0 + 16 * t + cl;
      double vr = 0.0, vi = 0.0;
      for (int d = kq; d < p.nele; d += 4) {
        const int off = q >= qnew && q < p.nq ? (ldiag[d] * p.nq + q) * (CPLX ? 16 : 8) : -1;
        if (CPLX) {
          const double2 v = bload_d2(rw, off);
          vr += v.x;
          vi += v.y;
        } else {
          vr += load_d(rw, off);
        }
      }
      vr += __shfl_xor(vr, 16);
      vr += __shfl_xor(vr, 32);
      double* fold = wf + ((noff >> 2) * G + t) * kF + 16 * (noff & 3) + cl;
      if (kq == 0) fold[0] = vr;
      if (CPLX) {
        vi += __shfl_xor(vi, 16);
        vi += __shfl_xor(vi, 32);
        if (kq == 0) fold[64] = vi;
      }
    }
    if (tid < p.copies) turns[tid] = tid;
    __syncthreads();

    u32x4 ring[kPullDepth];
    // k step s of a tile; rows past the live ones and columns past the row
    // are out of range and read zero
    auto load_b = [&](int s, uint32_t o) {
      const uint32_t r = lrow[4 * s + kq];
      return __builtin_amdgcn_raw_buffer_load_b128(
          rc, static_cast<int>(r | o) < 0 ? -1 : static_cast<int>(r + o), 0, 0);
    };
    auto column = [&](int tile) {
      const int jb = tile * 16 + cl;
      return jb < lenb ? static_cast<uint32_t>(jb) * 16u : kPullNoRow;
    };
    if (wave < ntile) {
#pragma unroll
      for (int j = 0; j < kPullDepth; ++j) ring[j] = load_b(j, column(wave));
    }
    for (int tile = wave; tile < ntile; tile += nwave) {
      const int jb = tile * 16 + cl;
      const uint32_t o = column(tile);
      // target words, volatile so that the loads stay ahead of the products
      uint32_t fv[G][4];
      const int fo = jb < lenb ? (kq * lenb + jb) * 4 : -1;
#pragma unroll
      for (int t = 0; t < G; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          fv[t][e] = __builtin_amdgcn_raw_buffer_load_b32(
              rf, fo, (q0 + 16 * t + 4 * e) * 4 * lenb, kVolatile);
        }
      double4_t zr[G], zi[G];
#pragma unroll
      for (int t = 0; t < G; ++t) {
        zr[t] = double4_t{0, 0, 0, 0};
        zi[t] = double4_t{0, 0, 0, 0};
      }
      // A of step s + 1 is read while step s multiplies
      double ar[2][G], ai[2][G];
      auto load_a = [&](int s, double (&r)[G], double (&im)[G]) {
        const double* f = wf + (s < ks ? s : 0) * (G * kF) + lane;
#pragma unroll
        for (int t = 0; t < G; ++t) {
          r[t] = f[t * kF];
          if (CPLX) im[t] = f[t * kF + 64];
        }
      };
      auto step = [&](u32x4 bv, const double (&r)[G], const double (&im)[G]) {
        const double br = u2d(bv[0], bv[1]);
        const double bi = u2d(bv[2], bv[3]);
#pragma unroll
        for (int t = 0; t < G; ++t) {
          zr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[t], br, zr[t], 0, 0, 0);
          zi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(r[t], bi, zi[t], 0, 0, 0);
        }
        if (CPLX) {
#pragma unroll
          for (int t = 0; t < G; ++t) {
            zr[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(-im[t], bi, zr[t], 0, 0, 0);
            zi[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(im[t], br, zi[t], 0, 0, 0);
          }
        }
      };
      load_a(0, ar[0], ai[0]);
      int s0 = 0;
      for (; s0 + kPullDepth <= ks; s0 += kPullDepth) {
#pragma unroll
        for (int j = 0; j < kPullDepth; ++j) {
          load_a(s0 + j + 1, ar[(j + 1) & 1], ai[(j + 1) & 1]);
          step(ring[j], ar[j & 1], ai[j & 1]);
          ring[j] = load_b(s0 + j + kPullDepth, o);
        }
      }
#pragma unroll
      for (int j = 0; j < kPullDepth - 1; ++j)
        if (s0 + j < ks) {
          load_a(s0 + j + 1, ar[(j + 1) & 1], ai[(j + 1) & 1]);
          step(ring[j], ar[j & 1], ai[j & 1]);
        }
      // the next tile's first steps are in flight during the additions
      if (tile + nwave < ntile) {
#pragma unroll
        for (int j = 0; j < kPullDepth; ++j) ring[j] = load_b(j, column(tile + nwave));
      }
      // the rows' adders ahead of the waves that multiply
      __builtin_amdgcn_s_setprio(2);
      if (p.copies < nwave)
        while (__builtin_amdgcn_readfirstlane(__hip_atomic_load(
                   turn, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != tile)
          __builtin_amdgcn_s_sleep(1);
      asm volatile("" ::: "memory");
#pragma unroll
      for (int t = 0; t < G; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t f = fv[t][e];
          if (f) {
            double* to = reinterpret_cast<double*>(accum + (f << 1));
            const uint32_t sg = f & 0x80000000u;
            __hip_atomic_fetch_add(to, with_sign(zr[t][e], sg), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(to + 1, with_sign(zi[t][e], sg), __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
          }
        }
      if (p.copies < nwave) {
        // this tile's additions are done before the next one's begin
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (lane == 0)
          __hip_atomic_store(turn, tile + p.copies, __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_WORKGROUP);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
  }
  double2* racc = reinterpret_cast<double2*>(p.rowacc) + ia * p.lenb;
  double sq = 0.0;
  for (int x = tid; x < lenb; x += nt) {
    double re = 0.0, im = 0.0;
    if (!p.ha) {
      const double2 r = racc[x];
      re = r.x;
      im = r.y;
    }
    for (int c = 0; c < p.copies; ++c) {
      const double2 v = accs[c * lenb + x];
      re += v.x;
      im += v.y;
    }
    if (!p.out) {
      racc[x] = make_double2(re, im);
      continue;
    }
    const int64_t idx = ia * p.lenb + x;
    double vr = p.alpha_re * re - p.alpha_im * im;
    double vi = p.alpha_re * im + p.alpha_im * re;
    if (p.beta_re != 0.0 || p.beta_im != 0.0) {
      const double2 c = reinterpret_cast<const double2*>(p.cin)[idx];
      vr += p.beta_re * c.x - p.beta_im * c.y;
      vi += p.beta_re * c.y + p.beta_im * c.x;
    }
    reinterpret_cast<double2*>(p.out)[idx] = make_double2(vr, vi);
    sq += vr * vr + vi * vi;
    if (p.acc) {
      double2* a = reinterpret_cast<double2*>(p.acc) + idx;
      const double2 o = p.acc0 ? reinterpret_cast<const double2*>(p.acc0)[idx] : *a;
      *a = make_double2(o.x + vr, o.y + vi);
    }
  }
  if (p.partials) row_norm(sq, p.partials + ia, smem);
}

template <bool CPLX, int G>
__global__ void __launch_bounds__(512, 2) k_pull_rows_f64(PullArgs p) {
  extern __shared__ __align__(16) char smem[];
  if (p.done && *p.done) return;
  if (p.series.partials && series_done(p.series, static_cast<int>(p.lena))) return;
  pull_row<CPLX, G>(p, xcd_order(blockIdx.x, p.lena), smem);
}

// One Taylor step of every sector of a batch group (sectors of G W tiles, real
// operators, 4-wave workgroups).  Step 0 is apply_out = H C0; step k >= 1 is
// term_k = alpha H term_(k-1), result += term_k (step 1: result = C0 + term_1),
// with the terms alternating between two buffers, so no copy and no second
// pass is needed.  Small sectors are bound by launches and idle CUs: a step of
// one is 2 launches of ~10 us for a handful of workgroups.  30 random sectors
// of 4 to 12 orbitals, one apply and 10 terms: 3602 us with each sector's own
// launches (one in-place apply per term), 1229 us with the groups (2749 us
// with the push-form row groups before the pull form).
struct PullGroupSector {
  PullArgs args;                           // coeff, out, acc per step
  const double* ha;
  const double* hb;
  const double* coeff0;
  double* apply_out;
  double* term[2];
  double* result;
  int row0, tile0, ta, tb;                 // first workgroup of each kernel
};

__device__ __forceinline__ int group_find(const PullGroupSector* secs, int nsec,
                                          int block, bool rows) {
  int lo = 0, hi = nsec - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((rows ? secs[mid].row0 : secs[mid].tile0) <= block) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

__device__ __forceinline__ const double* group_source(const PullGroupSector& s, int step) {
  return step <= 1 ? s.coeff0 : s.term[step & 1];
}

__global__ void __launch_bounds__(256, 4)
k_same_spin_group(const PullGroupSector* __restrict__ secs, int nsec, int step) {
  __shared__ double2 red[4 * 256];
  const int i = group_find(secs, nsec, blockIdx.x, false);
  const PullGroupSector& s = secs[i];
  if (step == 0 && !s.apply_out) return;
  same_spin_tile<false, 1, 1, true>(blockIdx.x - s.tile0, s.args.lena, s.args.lenb, s.ha,
                              s.hb, group_source(s, step), s.args.rowacc, s.ta, s.tb, red);
}

template <int G>
__global__ void __launch_bounds__(256, 2)
k_pull_rows_group(const PullGroupSector* __restrict__ secs, int nsec, int step,
                  double alpha_re, double alpha_im) {
  extern __shared__ __align__(16) char smem[];
  const int i = group_find(secs, nsec, blockIdx.x, true);
  const PullGroupSector& s = secs[i];
  PullArgs p = s.args;
  p.coeff = group_source(s, step);
  p.out = step == 0 ? s.apply_out : s.term[(step + 1) & 1];
  if (!p.out) return;
  p.alpha_re = step == 0 ? 1.0 : alpha_re;
  p.alpha_im = step == 0 ? 0.0 : alpha_im;
  p.acc = step == 0 ? nullptr : s.result;
  p.acc0 = step == 1 ? s.coeff0 : nullptr;
  pull_row<false, G>(p, blockIdx.x - s.row0, smem);
}

// Target words of the row kernel from a forward table: 8 (target + 1), bit 31
// the sign; 0 where the excitation vanishes.  (word << 1) is the byte offset
// of accumulator target + 1.
__global__ void __launch_bounds__(256)
k_pull_table(int64_t n, int64_t padded, const int32_t* __restrict__ fwd,
             uint32_t* __restrict__ tab) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= padded) return;
  const int32_t f = i < n ? fwd[i] : 0;
  tab[i] = static_cast<uint32_t>(iabs(f)) << 3 | (f < 0 ? 0x80000000u : 0u);
}

// Whether the same-spin product splits its sums (see launch_same_spin).
bool split_same_spin(int64_t lena, int64_t lenb) {
  return (lena + 63) / 64 * ((lenb + 63) / 64) < 150;
}

// Whether the rows compute their same-spin part themselves: it saves a launch,
// but every row reads all of C and Hbb, in time about lenb max(lena, lenb).
// Evolution in us, same-spin kernel / in the row: 20 x 15 strings 449 / 339,
// 35 x 35 420 / 346, 56 x 56 432 / 386, 70 x 70 505 / 500, 126 x 84 502 / 551,
// 252 x 45 533 / 590.  The line lies at the tie (4900); nothing between it and
// 10584 was measured.
bool pull_in_row(int64_t lena, int64_t lenb) {
  return lenb * (lena > lenb ? lena : lenb) <= kInRowMax && lena <= 256;
}

// How a sector runs: W tiles per pass, waves, accumulator rows.
struct PullPlan {
  int ks, tiles, pass, copies, threads;
  size_t lds;
};

// False if not even one W tile fits beside one accumulator row.
bool pull_plan(bool cplx, int noff, int64_t lenb, int nq, PullPlan* pl) {
  const int ks = (noff + 1 + 3) / 4;
  const int nqt = (nq + 15) / 16;
  int g = nqt < kPullTiles ? nqt : kPullTiles;
  while (g > 0 && pull_lds_bytes(cplx, ks, lenb, g, 1) > kLdsLimit) --g;
  if (g <= 0) return false;
  pl->ks = ks;
  pl->pass = (nqt + g - 1) / g;
  pl->tiles = (nqt + pl->pass - 1) / pl->pass;
  // two 4-wave workgroups per CU while their LDS fits, else one of 8 waves;
  // as many accumulator rows as the rest of that LDS holds
  const bool two = pull_lds_bytes(cplx, ks, lenb, pl->tiles, 1) <= kLdsLimit / 2;
  const size_t limit = two ? kLdsLimit / 2 : kLdsLimit;
  pl->threads = two ? 256 : 512;
  pl->copies = 1;
  while (2 * pl->copies * 64 <= pl->threads &&
         pull_lds_bytes(cplx, ks, lenb, pl->tiles, 2 * pl->copies) <= limit)
    pl->copies *= 2;
  pl->lds = pull_lds_bytes(cplx, ks, lenb, pl->tiles, pl->copies);
  return true;
}

template <bool CPLX>
int launch_rows(const PullPlan& pl, const PullArgs& p, hipStream_t st) {
  const unsigned grid = static_cast<unsigned>(p.lena);
  switch (pl.tiles) {
#define FQEHIP_PULL_CASE(N)                                            \
  case N:                                                              \
    k_pull_rows_f64<CPLX, N><<<grid, pl.threads, pl.lds, st>>>(p);     \
    break;
    FQEHIP_PULL_CASE(1)
    FQEHIP_PULL_CASE(2)
    FQEHIP_PULL_CASE(3)
    FQEHIP_PULL_CASE(4)
    FQEHIP_PULL_CASE(5)
    FQEHIP_PULL_CASE(6)
    FQEHIP_PULL_CASE(7)
#undef FQEHIP_PULL_CASE
    default:
      set_error("k_pull_rows_f64: %d tiles", pl.tiles);
      return FQEHIP_ERR_INVALID;
  }
  FQEHIP_CHECK_LAUNCH("k_pull_rows_f64");
  return FQEHIP_OK;
}

}  // namespace

// The limits are those of a complex operator (the narrower ones), so that
// the answer is the sector's alone.
static bool pull_limits(const fqehip_sector* s) {
  const int noff = s->nalpha * (s->norb - s->nalpha);
  PullPlan pl;
  return s->npull > 0 && s->lena > 0 && s->lenb > 0 &&
         s->nalpha * (s->norb - s->nalpha + 1) <= 64 && noff < kPullMaxK &&
         s->lena * s->lenb * 16 < kOffLimit && s->lena * s->lena * 16 < kOffLimit &&
         s->lenb * s->lenb * 16 < kOffLimit &&
         static_cast<int64_t>(s->npull + 15) * s->lenb * 4 < kOffLimit &&
         pull_plan(true, noff, s->lenb, s->npull, &pl);
}

bool pull_supported(const fqehip_sector* s) {
  return s->pull_w && s->haa && s->hbb && s->dexc_a && s->pull_fwd && pull_limits(s);
}

bool pull_one_launch(const fqehip_sector* s) {
  return pull_in_row(s->lena, s->lenb);
}

// rowacc = Haa C + C Hbb^T (complex128, 16 lena lenb bytes).
int launch_same_spin(const fqehip_sector* s, int complex_op,
                     const double* coeff, double* rowacc,
                     const PullSeries& series, hipStream_t st,
                     const int32_t* done) {
  // tiles of 64 x 128 (64 x 64 complex operators) once they give every CU two
  // workgroups; 32 x 64 from 300 workgroups on (924 x 924 strings: 0.126 ms,
  // 0.149 with 64 x 64); below, 16 x 16 with the sums split over the waves
  // (split / 32 x 64, ms: 924 x 924 0.164 / 0.128, 792 x 792 0.131 / 0.117, 715 x
  // 715 0.083 / 0.099, 792 x 495 0.061 / 0.071)
  const int64_t l = s->lena, m = s->lenb;
  const bool large = (l + 63) / 64 * ((m + (complex_op ? 63 : 127)) / (complex_op ? 64 : 128)) >= 512;
  const bool mid = !large && !split_same_spin(l, m);
  if (complex_op) {
    if (large) same_spin<true, 2, 2>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
    else if (mid) same_spin<true, 1, 2>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
    else same_spin<true, 1, 1, true>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
  } else {
    if (large) same_spin<false, 2, 4>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
    else if (mid) same_spin<false, 1, 2>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
    else same_spin<false, 1, 1, true>(l, m, s->haa, s->hbb, coeff, rowacc, series, st, done);
  }
  FQEHIP_CHECK_LAUNCH("k_same_spin_f64");
  return FQEHIP_OK;
}

namespace {

// The sector's part of the row kernel's arguments.
bool pull_args(const fqehip_sector* s, int complex_op, PullArgs* p, PullPlan* pl) {
  if (!pull_plan(complex_op != 0, s->nalpha * (s->norb - s->nalpha), s->lenb,
                 s->npull, pl)) {
    set_error("k_pull_rows_f64: lenb=%lld does not fit in LDS",
              static_cast<long long>(s->lenb));
    return false;
  }
  *p = PullArgs{};
  p->norb = s->norb;
  p->compressed = s->npull == s->norb * (s->norb + 1) / 2 ? 1 : 0;
  p->nele = s->nalpha;
  p->nq = s->npull;
  p->lena = s->lena;
  p->lenb = s->lenb;
  p->ks = pl->ks;
  p->pass = pl->pass;
  p->copies = pl->copies;
  p->w = s->pull_w;
  p->dexc = s->dexc_a;
  p->fwd = s->pull_fwd;
  if (pull_in_row(s->lena, s->lenb)) {
    p->ha = s->haa;
    p->hb = s->hbb;
  }
  return true;
}

}  // namespace

// The opposite-spin rows on top of rowacc; with e.out set also the epilogue
// out = alpha (H C) + beta cin, acc += out, partials[ia] = |out row|^2 (out must
// not alias coeff: other workgroups still read it).
int launch_pull_rows(const fqehip_sector* s, int complex_op,
                     const double* coeff, double* rowacc,
                     const PullEpilogue& e, hipStream_t st, const int32_t* done) {
  PullPlan pl;
  PullArgs p;
  if (!pull_args(s, complex_op, &p, &pl)) return FQEHIP_ERR_INVALID;
  p.coeff = coeff;
  p.rowacc = rowacc;
  p.alpha_re = e.alpha_re;
  p.alpha_im = e.alpha_im;
  p.beta_re = e.beta_re;
  p.beta_im = e.beta_im;
  p.cin = e.cin;
  p.out = e.out;
  p.acc = e.acc;
  p.partials = e.partials;
  p.series = e.series;
  p.done = done;
  return complex_op ? launch_rows<true>(pl, p, st) : launch_rows<false>(pl, p, st);
}

// Batch groups.  The class of a sector is the W tile count its rows run with
// (1..7); 0 for sectors that keep their own launches: 8-wave workgroups and
// same-spin products past the split tile.
int pull_group_class(const fqehip_sector* s) {
  PullPlan pl;
  if (!pull_plan(false, s->nalpha * (s->norb - s->nalpha), s->lenb, s->npull, &pl) ||
      pl.threads != 256 || !split_same_spin(s->lena, s->lenb))
    return 0;
  return pl.tiles;
}

size_t pull_group_bytes(int nsec) { return nsec * sizeof(PullGroupSector); }

// Fills host descriptors for the items of one class; rowacc and the second
// term buffer from each item's workspace (spare: byte offset of the latter).
int pull_group_fill(const fqehip_batch_item* const* items, const int64_t* spare,
                    int nsec, void* host, PullGroupLaunch* g) {
  PullGroupSector* secs = static_cast<PullGroupSector*>(host);
  *g = PullGroupLaunch{};
  g->nsec = nsec;
  for (int i = 0; i < nsec; ++i) {
    const fqehip_batch_item& it = *items[i];
    const fqehip_sector& sc = it.sector;
    PullGroupSector& o = secs[i];
    o = PullGroupSector{};
    PullPlan pl;
    if (!pull_args(&sc, 0, &o.args, &pl)) return FQEHIP_ERR_INVALID;
    o.args.rowacc = static_cast<double*>(it.d_workspace);
    o.ha = sc.haa;
    o.hb = sc.hbb;
    o.coeff0 = static_cast<const double*>(it.d_coeff0);
    o.apply_out = static_cast<double*>(it.d_apply_out);
    o.term[0] = static_cast<double*>(it.d_term);
    o.term[1] = reinterpret_cast<double*>(static_cast<char*>(it.d_workspace) + spare[i]);
    o.result = it.d_result;
    o.row0 = g->rows;
    o.tile0 = g->tiles;
    if (!o.args.ha) {
      o.ta = static_cast<int>((sc.lena + 15) / 16);
      o.tb = static_cast<int>((sc.lenb + 15) / 16);
    }
    g->rows += static_cast<int>(sc.lena);
    g->tiles += o.ta * o.tb;
    g->cls = pl.tiles;
    g->lds = pl.lds > g->lds ? pl.lds : g->lds;
    g->any_apply = g->any_apply || it.d_apply_out != nullptr;
  }
  return FQEHIP_OK;
}

// Step `step` of the group: the same-spin products, then the rows.
int launch_pull_group(const PullGroupLaunch& g, const void* d_secs, int step,
                      double ar, double ai, hipStream_t st) {
  const PullGroupSector* secs = static_cast<const PullGroupSector*>(d_secs);
  if (g.tiles > 0) {
    k_same_spin_group<<<g.tiles, 256, 0, st>>>(secs, g.nsec, step);
    FQEHIP_CHECK_LAUNCH("k_same_spin_group");
  }
  switch (g.cls) {
#define FQEHIP_PULL_CASE(N)                                                  \
  case N:                                                                    \
    k_pull_rows_group<N><<<g.rows, 256, g.lds, st>>>(secs, g.nsec, step, ar, ai); \
    break;
    FQEHIP_PULL_CASE(1)
    FQEHIP_PULL_CASE(2)
    FQEHIP_PULL_CASE(3)
    FQEHIP_PULL_CASE(4)
    FQEHIP_PULL_CASE(5)
    FQEHIP_PULL_CASE(6)
    FQEHIP_PULL_CASE(7)
#undef FQEHIP_PULL_CASE
    default:
      set_error("k_pull_rows_group: class %d", g.cls);
      return FQEHIP_ERR_INVALID;
  }
  FQEHIP_CHECK_LAUNCH("k_pull_rows_group");
  return FQEHIP_OK;
}

}  // namespace fqehip

using namespace fqehip;

extern "C" int fqehip_pull_fits_supported(const fqehip_sector* s, int complex_op) {
  if (!s || s->norb <= 0 || !pull_limits(s)) return 0;
  // the columns of Haa and Hbb in LDS (fqehip_spin_block)
  const int64_t longest = s->lena > s->lenb ? s->lena : s->lenb;
  return (longest + s->npull) * (complex_op ? 16 : 8) <= static_cast<int64_t>(kLdsLimit);
}

extern "C" int64_t fqehip_pull_table_count(const fqehip_sector* s, int complex_op) {
  PullPlan pl;
  if (!s || s->npull <= 0 || s->lenb <= 0 ||
      !pull_plan(complex_op != 0, s->nalpha * (s->norb - s->nalpha), s->lenb,
                 s->npull, &pl))
    return -1;
  // as the row kernel walks them: 16 rows of every tile of every pass
  int end = 0;
  for (int ps = 0; ps < pl.pass; ++ps) {
    const int q0 = pull_pass_start(ps, pl.tiles, s->npull);
    if (q0 < 0 || q0 > end) return -1;
    end = q0 + 16 * pl.tiles;
  }
  return static_cast<int64_t>(end) * s->lenb;
}

extern "C" int fqehip_pull_table(int npair, int64_t len, const int32_t* d_fwd,
                                 uint32_t* d_tab, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(npair >= 0 && len >= 0 && len < (1 << 27), "npair=%d len=%lld",
                   npair, static_cast<long long>(len));
  const int64_t n = npair * len;
  const int64_t padded = (npair + 15) / 16 * 16 * len;
  if (n == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_fwd && d_tab, "NULL pointer");
  k_pull_table<<<blocks_for(padded, 256), 256, 0, as_stream(stream)>>>(n, padded, d_fwd,
                                                                       d_tab);
  FQEHIP_CHECK_LAUNCH("k_pull_table");
  return FQEHIP_OK;
}
