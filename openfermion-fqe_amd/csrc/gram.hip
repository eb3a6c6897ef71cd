// Complex Gram matrix G[p][q] = sum_i conj(A[p][i]) B[q][i] of two blocks of
// k complex128 vectors (k rows, n interleaved complex entries each) on the
// FP64 matrix cores: the 2-RDM's dvec overlap D2^H D
// (reference src/fqe/fqe_data.py:1767-1782, tensordot of dvec2.conj() and
// dvec over the determinant axes).
//
// With A = X + iY and B = U + iV:
//   Re G = X U^T + Y V^T,   Im G = X V^T - Y U^T,
// four v_mfma_f64_16x16x4f64 per 4-element step of i and 16 x 16 tile.  The
// matrix unit bounds it, so the tiling is there to keep operand traffic
// below it: a wave holds a 32 x 32 block (each operand register feeds two
// tiles; 16 bytes a clock and CU out of the caches), loads 8 elements of i at
// a time straight into the MFMA layout (any bijection of i to k works for a
// sum over i, so a lane takes two adjacent ones in 16-byte loads) and has the
// next 8 in flight.  The four waves of a workgroup take every fourth step of
// the same block and chunk of i, so their loads share cache lines, and are
// summed in LDS; a second kernel sums the chunks.  Both in a fixed order.
// With a == b only blocks on and above the diagonal are computed.
//
// 101 x 101 over 52920 elements (a 2-RDM at 10 orbitals, 5 + 4 electrons):
// 77 + 5 us (56 TFLOP/s of the computed blocks), against 470 us with 16 x 16
// tiles per wave, 8-byte loads and all blocks.
#include "fqehip_common.h"

namespace fqehip {
namespace {

typedef double double4_t __attribute__((ext_vector_type(4)));
// rows may start at any multiple of 8 bytes (planar rows of odd length)
typedef double double2u_t __attribute__((ext_vector_type(2), aligned(8)));

constexpr int kGBlock = 32;              // rows and columns of a block
constexpr int kGWaves = 4;
constexpr int kGStep = 8;                // i per wave step
constexpr int kGQuad = kGWaves * kGStep; // i per workgroup step
// workgroups that are resident at once (two per CU): one wave of them
constexpr int kGTarget = 512;

struct GramPlan {
  int blocks, pairs, nchunk;
  int64_t chunk;
};

GramPlan gram_plan(int64_t n, int k, bool hermitian) {
  GramPlan p;
  p.blocks = (k + kGBlock - 1) / kGBlock;
  p.pairs = hermitian ? p.blocks * (p.blocks + 1) / 2 : p.blocks * p.blocks;
  int64_t c = kGTarget / p.pairs;
  // at least 8 steps per wave
  const int64_t most = (n + 8 * kGQuad - 1) / (8 * kGQuad);
  c = c < 1 ? 1 : (c > most ? most : c);
  p.chunk = ((n + c - 1) / c + kGQuad - 1) / kGQuad * kGQuad;
  p.nchunk = static_cast<int>((n + p.chunk - 1) / p.chunk);
  return p;
}

// Block (bp, bq) of pair index t; bp <= bq row by row if hermitian.
__device__ __forceinline__ void gram_block(int t, int blocks, bool hermitian,
                                           int* bp, int* bq) {
  int r = 0;
  if (!hermitian) {
    r = t / blocks;
    *bp = r;
    *bq = t - r * blocks;
    return;
  }
  while (t >= blocks - r) {
    t -= blocks - r;
    ++r;
  }
  *bp = r;
  *bq = r + t;
}

// Two adjacent elements of a row: re[0..1], im[0..1].  PLANAR rows hold n real
// parts, then n imaginary parts; the others interleave them.
template <bool PLANAR>
__device__ __forceinline__ void gram_load(const double* row, int64_t n, int64_t i,
                                          double (&re)[2], double (&im)[2]) {
  const double* a = PLANAR ? row + i : row + 2 * i;
  const double2u_t u = *reinterpret_cast<const double2u_t*>(a);
  const double2u_t v = *reinterpret_cast<const double2u_t*>(a + (PLANAR ? n : 2));
  re[0] = u[0];
  re[1] = PLANAR ? u[1] : v[0];
  im[0] = PLANAR ? v[0] : u[1];
  im[1] = v[1];
}

// The same with elements at and past `end` zero.
template <bool PLANAR>
__device__ __forceinline__ void gram_load_tail(const double* row, int64_t n, int64_t i,
                                               int64_t end, double (&re)[2],
                                               double (&im)[2]) {
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const bool ok = i + e < end;
    re[e] = ok ? (PLANAR ? row[i + e] : row[2 * (i + e)]) : 0.0;
    im[e] = ok ? (PLANAR ? row[n + i + e] : row[2 * (i + e) + 1]) : 0.0;
  }
}

// grid.x: block pairs, grid.y: chunks of i
template <bool PLANAR>
__global__ void __launch_bounds__(kGWaves * 64, 2)
k_gram_f64(int64_t n, int k, int blocks, bool hermitian, int64_t chunk,
           const double* __restrict__ a, const double* __restrict__ b,
           double* __restrict__ part) {
  __shared__ double red[kGBlock * kGBlock * 2];
  const int wave = threadIdx.x >> 6;
  const int lane = threadIdx.x & 63;
  const int r16 = lane & 15;
  int bp, bq;
  gram_block(blockIdx.x, blocks, hermitian, &bp, &bq);
  const int64_t i0 = blockIdx.y * chunk;
  const int64_t i1 = i0 + chunk < n ? i0 + chunk : n;
  // rows past k read row 0; their products are not stored
  const double *ap[2], *bp_[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int p = bp * kGBlock + 16 * t + r16;
    const int q = bq * kGBlock + 16 * t + r16;
    ap[t] = a + 2 * n * static_cast<int64_t>(p < k ? p : 0);
    bp_[t] = b + 2 * n * static_cast<int64_t>(q < k ? q : 0);
  }
  double4_t re[2][2], im[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      re[x][y] = double4_t{0, 0, 0, 0};
      im[x][y] = double4_t{0, 0, 0, 0};
    }
  struct Step {
    double xr[2][2], xi[2][2], ur[2][2], ui[2][2];
  };
  auto products = [&](const Step& s) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) {
          re[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.xr[x][e], s.ur[y][e], re[x][y], 0, 0, 0);
          im[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.xr[x][e], s.ui[y][e], im[x][y], 0, 0, 0);
          re[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(s.xi[x][e], s.ui[y][e], re[x][y], 0, 0, 0);
          im[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(-s.xi[x][e], s.ur[y][e], im[x][y], 0, 0, 0);
        }
  };
  // operand layout: A[row l % 16][k l / 16], B[k l / 16][column l % 16]
  const int64_t first = i0 + wave * kGStep + 2 * (lane >> 4);
  auto load = [&](Step& s, int64_t i) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      gram_load<PLANAR>(ap[t], n, i, s.xr[t], s.xi[t]);
      gram_load<PLANAR>(bp_[t], n, i, s.ur[t], s.ui[t]);
    }
  };
  // full steps of this wave (the same for all of its lanes)
  const int64_t left = i1 - i0 - wave * kGStep;
  const int nfull = left < kGStep ? 0 : static_cast<int>((left - kGStep) / kGQuad) + 1;
  if (nfull) {
    Step s[2];
    load(s[0], first);
    int j = 0;
    for (; j + 2 <= nfull; j += 2) {
      load(s[1], first + static_cast<int64_t>(j + 1) * kGQuad);
      products(s[0]);
      load(s[0], first + static_cast<int64_t>(j + 2 < nfull ? j + 2 : j) * kGQuad);
      products(s[1]);
    }
    if (j < nfull) products(s[0]);
  }
  const int64_t tail = left - static_cast<int64_t>(nfull) * kGQuad;
  if (tail > 0) {                          // fewer than kGStep elements
    const int64_t i = first + static_cast<int64_t>(nfull) * kGQuad;
    Step s;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      gram_load_tail<PLANAR>(ap[t], n, i, i1, s.xr[t], s.xi[t]);
      gram_load_tail<PLANAR>(bp_[t], n, i, i1, s.ur[t], s.ui[t]);
    }
    products(s);
  }
  // waves 1..3 one after the other on top of each other's sums, wave 0 last
  // and out.  Item j of lane l is row l / 16 + 4 j, column l % 16.
  double* dst = part + (static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x) *
                           (kGBlock * kGBlock * 2);
  for (int w = kGWaves - 1; w >= 0; --w) {
    if (wave == w) {
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const int at = ((16 * x + (lane >> 4) + 4 * j) * kGBlock + 16 * y + r16) * 2;
            double vr = re[x][y][j], vi = im[x][y][j];
            if (w < kGWaves - 1) {
              vr += red[at];
              vi += red[at + 1];
            }
            if (w) {
              red[at] = vr;
              red[at + 1] = vi;
            } else {
              *reinterpret_cast<double2*>(dst + at) = make_double2(vr, vi);
            }
          }
    }
    __syncthreads();
  }
}

// Sums the chunks of each block element and places it (and, for a hermitian
// product, its conjugate).  grid.x: block pairs x 4 quarters of a block.
__global__ void __launch_bounds__(256)
k_gram_reduce(int k, int blocks, int pairs, bool hermitian, int nchunk,
              const double* __restrict__ part, double* __restrict__ out) {
  const int pair = blockIdx.x >> 2;
  const int x = (blockIdx.x & 3) * 256 + threadIdx.x;
  int bp, bq;
  gram_block(pair, blocks, hermitian, &bp, &bq);
  const int p = bp * kGBlock + x / kGBlock;
  const int q = bq * kGBlock + x % kGBlock;
  if (p >= k || q >= k) return;
  const double2* src = reinterpret_cast<const double2*>(part) +
                       static_cast<int64_t>(pair) * kGBlock * kGBlock + x;
  const int64_t pitch = static_cast<int64_t>(pairs) * kGBlock * kGBlock;
  double re = 0.0, im = 0.0;
#pragma unroll 8
  for (int c = 0; c < nchunk; ++c) {
    const double2 v = src[c * pitch];
    re += v.x;
    im += v.y;
  }
  double2* o = reinterpret_cast<double2*>(out);
  o[static_cast<int64_t>(p) * k + q] = make_double2(re, im);
  if (hermitian && bp != bq)
    o[static_cast<int64_t>(q) * k + p] = make_double2(re, -im);
}

__global__ void __launch_bounds__(256)
k_gram_zero(int64_t count, double* __restrict__ out) {
  const int64_t x = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (x < count) out[x] = 0.0;
}

template <bool PLANAR>
int gram(int64_t n, int k, const double* d_a, const double* d_b, double* d_out,
         double* d_workspace, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(n >= 0 && k >= 0 && k <= 4096, "n=%lld k=%d",
                   static_cast<long long>(n), k);
  if (k == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_out != nullptr, "NULL output");
  hipStream_t st = as_stream(stream);
  if (n == 0) {
    // an empty sum: zero the output with a kernel (no memset nodes)
    const int64_t kk2 = static_cast<int64_t>(k) * k * 2;
    k_gram_zero<<<blocks_for(kk2, 256), 256, 0, st>>>(kk2, d_out);
    FQEHIP_CHECK_LAUNCH("k_gram_zero");
    return FQEHIP_OK;
  }
  FQEHIP_CHECK_ARG(d_a && d_b && d_workspace, "NULL pointer");
  // the limit of one pass, from the 65535 chunks of 4096 it once had
  FQEHIP_CHECK_ARG((n + 4095) / 4096 <= 65535, "n=%lld too large for one Gram pass",
                   static_cast<long long>(n));
  const bool herm = d_a == d_b;
  const GramPlan pl = gram_plan(n, k, herm);
  k_gram_f64<PLANAR><<<dim3(pl.pairs, pl.nchunk), kGWaves * 64, 0, st>>>(
      n, k, pl.blocks, herm, pl.chunk, d_a, d_b, d_workspace);
  FQEHIP_CHECK_LAUNCH("k_gram_f64");
  k_gram_reduce<<<4 * pl.pairs, 256, 0, st>>>(k, pl.blocks, pl.pairs, herm,
                                              pl.nchunk, d_workspace, d_out);
  FQEHIP_CHECK_LAUNCH("k_gram_reduce");
  return FQEHIP_OK;
}

}  // namespace
}  // namespace fqehip

using namespace fqehip;

extern "C" int64_t fqehip_gram_workspace_bytes(int64_t n, int k) {
  if (n <= 0 || k <= 0) return 0;
  // the larger of the general and the hermitian plan
  int64_t most = 0;
  for (bool herm : {false, true}) {
    const GramPlan pl = gram_plan(n, k, herm);
    const int64_t tiles = static_cast<int64_t>(pl.pairs) * pl.nchunk;
    most = tiles > most ? tiles : most;
  }
  return most * kGBlock * kGBlock * 2 * static_cast<int64_t>(sizeof(double));
}

extern "C" int fqehip_gram(int64_t n, int k, const double* d_a,
                           const double* d_b, double* d_out,
                           double* d_workspace, void* stream) {
  return gram<false>(n, k, d_a, d_b, d_out, d_workspace, stream);
}

extern "C" int fqehip_gram_planar(int64_t n, int k, const double* d_a,
                                  const double* d_b, double* d_out,
                                  double* d_workspace, void* stream) {
  return gram<true>(n, k, d_a, d_b, d_out, d_workspace, stream);
}
