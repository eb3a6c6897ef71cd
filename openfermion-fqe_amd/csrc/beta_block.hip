// Beta-beta block of a pair-symmetric real operator and its product with
// the CI matrix (mixed-precision split apply).
//
// For A[p][q] = A[q][p] (p, q < npair) the operator
//   H = sum_pq A[p][q] E_p E_q + sum_q A[npair][q] E_q,   E_p = E^a_p + E^b_p
// splits exactly into (alpha and beta pair operators commute)
//   H C = sum_p E^a_p ( [A (D^a + 2 D^b)][p] + A[npair][p] C )  +  C Hbb^T,
//   Hbb = sum_pq A[p][q] E^b_p E^b_q + sum_q A[npair][q] E^b_q  (lenb x lenb),
// so the per-row kernel only scatters alpha excitations and every beta
// excitation of the output becomes one dense GEMM with Hbb.  The reference
// makes the same same-spin / opposite-spin split in its lm kernels
// (src/fqe/lib/fqe_data.c:668-720 and :879-996).
//
//   k_spin_block:  Hbb column by column, its non-zero elements found through
//                  the beta forward table (one workgroup per source string);
//   k_beta_split:  transpose and split into bfloat16 hi + lo, zero-padded
//                  to ldh x ldh (ldh a multiple of 128);
//   k_beta_gemm_bf16x3: out[Ia][Ib'] = sum_Ib C[Ia][Ib] Hbb[Ib'][Ib] on
//                  v_mfma_f32_16x16x32_bf16 with the three-product split;
//   k_beta_gemm_f64: the same product for complex128 C on
//                  v_mfma_f64_16x16x4f64, from the FP64 columns of Hbb.
#include "fqehip_common.h"

namespace fqehip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef double double4_t __attribute__((ext_vector_type(4)));

constexpr int kBlockThreads = 256;

__device__ __forceinline__ __bf16 to_bf16(float x) {
  return static_cast<__bf16>(x);  // round to nearest even (v_cvt_pk_bf16_f32)
}

__device__ __forceinline__ float from_bf16(__bf16 h) {
  return __uint_as_float(static_cast<uint32_t>(__builtin_bit_cast(uint16_t, h))
                         << 16);
}

__device__ __forceinline__ int32_t iabs(int32_t v) { return v < 0 ? -v : v; }

// Column s of the block, sum_pq V[p][q] E_p E_q + sum_q h[q] E_q between the
// strings t and s, E_(ai) = a+_a a_i.  An element is non-zero for t = s and for
// strings one or two excitations away, and each is computed as a whole by the
// threads that own it (i, j occupied in s, a, b empty, i < j, a < b):
//   i -> a, j -> b:  V[bj][ai] + V[ai][bj] - V[bi][aj] - V[aj][bi], times the sign
//       of E_bj E_ai;
//   i -> a:  h[ai] + V[ai][ii] + V[aa][ai] + sum over the other k of V[kk][ai] +
//       V[ai][kk] - V[ki][ak] (k occupied) or V[ak][ki] (k empty), times the sign of
//       E_ai: the ways over an intermediate string, in either order;
//   t = s:  sum_k h[kk] + sum_kl V[kk][ll] + sum_ia V[ia][ai].
// A compressed pair stands for both of its excitations, of which one applies.
// V[p][q] is amat[p * lda + q], h[q] is h1[q]; CPLX: both in the real 2 x 2 block
// form (real part at [2p][2q], imaginary at [2p + 1][2q]).
//
// One workgroup per source string; the column is assembled in LDS (targets are
// scattered, 645 of 6435 at 15 orbitals) and written in one piece, so what
// bounds it is that write and, below some hundreds of strings, two dependent
// table lookups.  Every element has one order of additions: the same bits on
// every run.  6435 strings of 15 orbitals: 137 us, 3432 of 14: 49, against 636
// and 202 when the workgroup went through the pairs q one after the other with
// two barriers each (V[p][q] E_p added to the column for all p at once).
template <bool CPLX>
struct BlockValue {
  double re, im;
};
template <>
struct BlockValue<false> {
  double re;
};

constexpr int kBlockOrb = 32;               // orbitals at most

// Only the empty or the full shell, on one string: the excitations that do not
// vanish are the occupation numbers, whatever the order of the pairs.
template <bool CPLX>
__global__ void __launch_bounds__(64)
k_spin_block_one(int npair, const int32_t* __restrict__ fwd,
                 const double* __restrict__ amat, int64_t lda,
                 const double* __restrict__ h1, double* __restrict__ hcol) {
  constexpr int kW = CPLX ? 2 : 1;
  double re = 0.0, im = 0.0;
  for (int q = threadIdx.x; q < npair; q += 64) {
    if (!fwd[q]) continue;
    re += h1[kW * q];
    if (CPLX) im += h1[lda + kW * q];
    for (int p = 0; p < npair; ++p) {
      if (!fwd[p]) continue;
      const double* e = amat + static_cast<int64_t>(kW) * p * lda + kW * q;
      re += e[0];
      if (CPLX) im += e[lda];
    }
  }
#pragma unroll
  for (int m = 1; m < 64; m <<= 1) {
    re += __shfl_xor(re, m);
    im += __shfl_xor(im, m);
  }
  if (threadIdx.x == 0) {
    hcol[0] = re;
    if (CPLX) hcol[1] = im;
  }
}

// LDS of a column: the values, then the lists of occupied and empty orbitals
// and of their pairs (16 bits each).
size_t spin_block_lds(int norb, int64_t len, bool cplx) {
  // both shells' pairs: the most that any filling has
  return static_cast<size_t>(len) * (cplx ? 16 : 8) +
         (static_cast<size_t>(norb) * (norb - 1) / 2 + 2 * kBlockOrb) * 2;
}

template <bool CPLX>
__global__ void __launch_bounds__(kBlockThreads)
k_spin_block(int norb, int compressed, int64_t len, const int32_t* __restrict__ fwd,
             const double* __restrict__ amat, int64_t lda,
             const double* __restrict__ h1, double* __restrict__ hcol) {
  typedef BlockValue<CPLX> V;
  constexpr int kW = CPLX ? 2 : 1;            // rows and columns per pair
  extern __shared__ __align__(16) char block_smem[];
  V* col = reinterpret_cast<V*>(block_smem);
  uint16_t* occ = reinterpret_cast<uint16_t*>(col + len);
  uint16_t* emp = occ + kBlockOrb;
  uint16_t* pairs = emp + kBlockOrb;          // of occ, then of emp: low i, high j
  const int64_t s = blockIdx.x;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  auto pair = [&](int i, int j) { return compressed ? comp_pair(i, j) : i * norb + j; };
  auto jump = [&](int i, int j, int64_t from) { return fwd[pair(i, j) * len + from]; };
  // every wave finds the occupied orbitals for itself
  const uint32_t mask = static_cast<uint32_t>(
      __ballot(lane < norb && jump(lane < norb ? lane : 0, lane < norb ? lane : 0, s) != 0));
  const int no = __popc(mask), ne = norb - no;
  const int npo = no * (no - 1) / 2, npe = ne * (ne - 1) / 2;
  if (tid < norb) {
    const uint32_t below = (1u << tid) - 1u;
    if (mask >> tid & 1) occ[__popc(mask & below)] = static_cast<uint16_t>(tid);
    else emp[__popc(~mask & below)] = static_cast<uint16_t>(tid);
  }
  for (int64_t x = tid; x < len; x += kBlockThreads) col[x] = V{};
  __syncthreads();
  for (int x = tid; x < no * no + ne * ne; x += kBlockThreads) {
    const bool o = x < no * no;
    const int n = o ? no : ne, y = o ? x : x - no * no;
    const int i = y / n, j = y - i * n;
    if (i >= j) continue;
    const uint16_t* l = o ? occ : emp;
    pairs[(o ? 0 : npo) + i * (2 * n - i - 1) / 2 + j - i - 1] =
        static_cast<uint16_t>(l[i] | l[j] << 8);
  }
  __syncthreads();

  auto add = [&](V& v, double f, int p, int q) {
    const double* e = amat + static_cast<int64_t>(kW) * p * lda + kW * q;
    v.re += f * e[0];
    if constexpr (CPLX) v.im += f * e[lda];
  };
  auto add_h = [&](V& v, int q) {
    v.re += h1[kW * q];
    if constexpr (CPLX) v.im += h1[lda + kW * q];
  };
  auto put = [&](int32_t f, bool minus, V v) {    // at f's target with its sign
    const double sg = (f < 0) != minus ? -1.0 : 1.0;
    v.re *= sg;
    if constexpr (CPLX) v.im *= sg;
    col[iabs(f) - 1] = v;
  };
  for (int x = tid; x < npo * npe; x += kBlockThreads) {
    const int y = x / npe;
    const int ij = pairs[y], ab = pairs[npo + x - y * npe];
    const int i = ij & 255, j = ij >> 8, a = ab & 255, b = ab >> 8;
    const int32_t f1 = jump(a, i, s);
    const int32_t f2 = jump(b, j, iabs(f1) - 1);
    const int ai = pair(a, i), bj = pair(b, j), aj = pair(a, j), bi = pair(b, i);
    V v{};
    add(v, 1.0, bj, ai);
    add(v, 1.0, ai, bj);
    add(v, -1.0, bi, aj);
    add(v, -1.0, aj, bi);
    put(f2, f1 < 0, v);
  }
  // eight lanes to an element, every eighth k each
  auto sum8 = [&](V& v) {
#pragma unroll
    for (int m = 1; m < 8; m <<= 1) {
      v.re += __shfl_xor(v.re, m);
      if constexpr (CPLX) v.im += __shfl_xor(v.im, m);
    }
  };
  const int sub = tid & 7;
  for (int x0 = 0; x0 < no * ne; x0 += kBlockThreads / 8) {
    const int x = x0 + (tid >> 3);
    const bool ok = x < no * ne;
    const int i = ok ? occ[x / ne] : 0, a = ok ? emp[x % ne] : 0;
    const int ai = pair(a, i);
    V v{};
    if (ok) {
      if (sub == 0) add_h(v, ai);
      for (int k = sub; k < norb; k += 8) {
        const int kk = pair(k, k);
        if (k == i) {
          add(v, 1.0, ai, kk);
        } else if (k == a) {
          add(v, 1.0, kk, ai);
        } else if (mask >> k & 1) {
          add(v, 1.0, kk, ai);
          add(v, 1.0, ai, kk);
          add(v, -1.0, pair(k, i), pair(a, k));
        } else {
          add(v, 1.0, pair(a, k), pair(k, i));
        }
      }
    }
    sum8(v);
    if (ok && sub == 0) put(jump(a, i, s), false, v);
  }
  if (tid < 64) {
    V v{};
    for (int x = lane; x < no * norb; x += 64) {
      const int i = occ[x / norb], k = x % norb;
      if (mask >> k & 1) add(v, 1.0, pair(i, i), pair(k, k));
      else add(v, 1.0, pair(i, k), pair(k, i));
      if (k == i) add_h(v, pair(i, i));
    }
    sum8(v);
#pragma unroll
    for (int m = 8; m < 64; m <<= 1) {
      v.re += __shfl_xor(v.re, m);
      if constexpr (CPLX) v.im += __shfl_xor(v.im, m);
    }
    if (lane == 0) col[s] = v;
  }
  __syncthreads();
  V* dst = reinterpret_cast<V*>(hcol) + s * len;
  for (int64_t x = tid; x < len; x += kBlockThreads) dst[x] = col[x];
}

// The orbitals behind npair pairs on len > 1 strings of one spin:
// norb (norb + 1) / 2 compressed pairs or norb^2, and len a binomial of norb
// (36 pairs are both, of 8 and of 6 orbitals, but no other number of strings
// than one is).  False if there are none.
bool spin_block_orbitals(int npair, int64_t len, int* norb, int* compressed) {
  for (int n = 2; n <= kBlockOrb; ++n) {
    const bool c = npair == n * (n + 1) / 2;
    if (!c && npair != n * n) continue;
    int64_t binom = n;
    for (int k = 1; k < n; ++k) {
      if (binom == len) {
        *norb = n;
        *compressed = c ? 1 : 0;
        return true;
      }
      binom = binom * (n - k) / (k + 1);
    }
  }
  return false;
}

template <bool CPLX>
int spin_block(int npair, int64_t len, const int32_t* fwd, const double* amat,
               int64_t lda, const double* h1, double* hcol, hipStream_t st) {
  if (len == 1) {
    k_spin_block_one<CPLX><<<1, 64, 0, st>>>(npair, fwd, amat, lda, h1, hcol);
    FQEHIP_CHECK_LAUNCH("k_spin_block_one");
    return FQEHIP_OK;
  }
  int norb = 0, compressed = 0;
  if (!spin_block_orbitals(npair, len, &norb, &compressed)) {
    set_error("k_spin_block: no orbitals have %d pairs and %lld strings", npair,
              static_cast<long long>(len));
    return FQEHIP_ERR_INVALID;
  }
  k_spin_block<CPLX><<<static_cast<unsigned>(len), kBlockThreads,
                       spin_block_lds(norb, len, CPLX), st>>>(
      norb, compressed, len, fwd, amat, lda, h1, hcol);
  FQEHIP_CHECK_LAUNCH("k_spin_block");
  return FQEHIP_OK;
}

// hhi/hlo[r][c] = split(Hbb[r][c]) = split(hcol[c][r]); zero outside lenb.
__global__ void __launch_bounds__(256)
k_beta_split(int64_t lenb, int64_t ldh, const double* __restrict__ hcol,
             __bf16* __restrict__ hhi, __bf16* __restrict__ hlo) {
  __shared__ double tile[32][33];
  const int64_t r0 = static_cast<int64_t>(blockIdx.y) * 32;   // Hbb rows
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * 32;   // Hbb columns
  const int tx = threadIdx.x & 31;
  const int ty = threadIdx.x >> 5;                            // 0..7
  for (int y = ty; y < 32; y += 8) {
    const int64_t c = c0 + y;
    const int64_t r = r0 + tx;
    tile[y][tx] = (c < lenb && r < lenb) ? hcol[c * lenb + r] : 0.0;
  }
  __syncthreads();
  for (int y = ty; y < 32; y += 8) {
    const double v = tile[tx][y];                             // Hbb[r0+y][c0+tx]
    const __bf16 h = to_bf16(static_cast<float>(v));
    const __bf16 l = to_bf16(static_cast<float>(v - static_cast<double>(from_bf16(h))));
    const int64_t o = (r0 + y) * ldh + c0 + tx;
    hhi[o] = h;
    hlo[o] = l;
  }
}

// GEMM tile: 128 rows (alpha strings) x 128 columns (target beta strings)
// per workgroup of 4 waves in a 2 x 2 arrangement, 64 x 64 per wave, K
// (source beta strings) in steps of 32.  The complex FP32 C tile is split
// into bf16 hi/lo of its real and imaginary parts in LDS (the A operand);
// the Hbb operand is read straight from the split copies in global memory
// (lane l: row col0 + l%16, k 8*(l/16)..+7, 16 contiguous bytes).
constexpr int kGT = 128;                  // tile rows and columns
constexpr int kGK = 32;                   // K step
constexpr int kGStride = kGK + 8;         // bf16 per LDS row (conflict-free)
constexpr int kXcds = 8;                  // XCDs of an MI355X
constexpr int kGroupRows = 8;             // tile rows per group of the order

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p,
                                                       int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0,
                                           static_cast<int>(bytes), 0x00020000);
}

// XCD-aware tile order: workgroups are dealt to the 8 XCDs round-robin, so
// workgroup L runs on XCD L % 8.  Each XCD takes one contiguous run of
// tiles in a grouped order (kGroupRows tile rows at a time), so the C rows
// and Hbb rows it reads stay within its own L2.  Returns false for the
// padding workgroups past ta * tb.
__device__ __forceinline__ bool xcd_tile(int ta, int tb, int per_xcd,
                                         int* tile_a, int* tile_b) {
  const int xcd = static_cast<int>(blockIdx.x % kXcds);
  const int t = xcd * per_xcd + static_cast<int>(blockIdx.x / kXcds);
  if (t >= ta * tb) return false;
  const int grp = t / (kGroupRows * tb);
  const int rows_here = (ta - grp * kGroupRows) < kGroupRows
                            ? (ta - grp * kGroupRows) : kGroupRows;
  const int within = t - grp * kGroupRows * tb;
  *tile_a = grp * kGroupRows + within % rows_here;
  *tile_b = within / rows_here;
  return true;
}

__global__ void __launch_bounds__(256, 2)
k_beta_gemm_bf16x3(int64_t lena, int64_t lenb, int64_t ldh,
                   const __bf16* __restrict__ hhi,
                   const __bf16* __restrict__ hlo,
                   const float* __restrict__ coeff, float* __restrict__ out,
                   const int32_t* __restrict__ done, int ta, int tb,
                   int per_xcd) {
  // two buffers of the split C tile (hr, lr, hi, li): the next K step is
  // stored while the current one feeds the MFMAs (one barrier per step)
  __shared__ __align__(16) __bf16 sa[2][4][kGT * kGStride];
  if (done && *done) return;
  int tile_a, tile_b;
  if (!xcd_tile(ta, tb, per_xcd, &tile_a, &tile_b)) return;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int64_t a0 = static_cast<int64_t>(tile_a) * kGT;
  const int64_t b0 = static_cast<int64_t>(tile_b) * kGT;
  const int wa = (wave >> 1) * 64;        // wave row offset in the tile
  const int wb = (wave & 1) * 64;         // wave column offset
  const __amdgpu_buffer_rsrc_t rc = rsrc(coeff, lena * lenb * 2 * sizeof(float));
  const __amdgpu_buffer_rsrc_t rh = rsrc(hhi, ldh * ldh * 2);
  const __amdgpu_buffer_rsrc_t rl = rsrc(hlo, ldh * ldh * 2);

  // C loader: thread -> tile row tid/2, 16 complex values from k 16*(tid%2)
  const int lr = tid >> 1;
  const int lk = 16 * (tid & 1);
  const int64_t arow = a0 + lr;
  const bool rowok = arow < lena;
  float cv[32];
  auto load_c = [&](int64_t k0) {
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      const int64_t k = k0 + lk + 2 * v;
      const int off = (rowok && k < lenb)
                          ? static_cast<int>((arow * lenb + k) * 2 * sizeof(float)) : -1;
      u32x4 x;
      if (k + 1 < lenb) {
        x = __builtin_amdgcn_raw_buffer_load_b128(rc, off, 0, 0);
      } else {
        // last value of a row: a 16-byte load would reach into the next row
        const u32x2 y = __builtin_amdgcn_raw_buffer_load_b64(rc, off, 0, 0);
        x = u32x4{y[0], y[1], 0u, 0u};
      }
      cv[4 * v + 0] = __uint_as_float(x[0]);
      cv[4 * v + 1] = __uint_as_float(x[1]);
      cv[4 * v + 2] = __uint_as_float(x[2]);
      cv[4 * v + 3] = __uint_as_float(x[3]);
    }
  };
  auto store_c = [&](int buf) {
    bf16x8 hr0, lr0, hi0, li0, hr1, lr1, hi1, li1;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const float re = cv[2 * j], im = cv[2 * j + 1];
      const __bf16 h = to_bf16(re), g = to_bf16(im);
      const __bf16 l = to_bf16(re - from_bf16(h)), m = to_bf16(im - from_bf16(g));
      if (j < 8) { hr0[j] = h; lr0[j] = l; hi0[j] = g; li0[j] = m; }
      else { hr1[j - 8] = h; lr1[j - 8] = l; hi1[j - 8] = g; li1[j - 8] = m; }
    }
    const int o = lr * kGStride + lk;
    *reinterpret_cast<bf16x8*>(&sa[buf][0][o]) = hr0;
    *reinterpret_cast<bf16x8*>(&sa[buf][0][o + 8]) = hr1;
    *reinterpret_cast<bf16x8*>(&sa[buf][1][o]) = lr0;
    *reinterpret_cast<bf16x8*>(&sa[buf][1][o + 8]) = lr1;
    *reinterpret_cast<bf16x8*>(&sa[buf][2][o]) = hi0;
    *reinterpret_cast<bf16x8*>(&sa[buf][2][o + 8]) = hi1;
    *reinterpret_cast<bf16x8*>(&sa[buf][3][o]) = li0;
    *reinterpret_cast<bf16x8*>(&sa[buf][3][o + 8]) = li1;
  };
  // Hbb operand registers for one K step: 4 column tiles x (hi, lo)
  bf16x8 bh[4], bl[4];
  auto load_h = [&](int64_t k0) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int64_t row = b0 + wb + 16 * c + (lane & 15);  // < ldh (padded)
      const int off = static_cast<int>((row * ldh + k0 + 8 * (lane >> 4)) * 2);
      const u32x4 xh = __builtin_amdgcn_raw_buffer_load_b128(rh, off, 0, 0);
      const u32x4 xl = __builtin_amdgcn_raw_buffer_load_b128(rl, off, 0, 0);
      bh[c] = __builtin_bit_cast(bf16x8, xh);
      bl[c] = __builtin_bit_cast(bf16x8, xl);
    }
  };

  floatx4 accr[4][4], acci[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      accr[r][c] = floatx4{0, 0, 0, 0};
      acci[r][c] = floatx4{0, 0, 0, 0};
    }

  const int64_t nk = (lenb + kGK - 1) / kGK;
  load_c(0);
  store_c(0);
  if (nk > 1) load_c(kGK);                // step 1 in flight
  __syncthreads();
  for (int64_t ks = 0; ks < nk; ++ks) {
    const int64_t k0 = ks * kGK;
    const int cb = static_cast<int>(ks & 1);
    load_h(k0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int o = (wa + 16 * r + (lane & 15)) * kGStride + 8 * (lane >> 4);
      const bf16x8 ahr = *reinterpret_cast<const bf16x8*>(&sa[cb][0][o]);
      const bf16x8 alr = *reinterpret_cast<const bf16x8*>(&sa[cb][1][o]);
      const bf16x8 ahi = *reinterpret_cast<const bf16x8*>(&sa[cb][2][o]);
      const bf16x8 ali = *reinterpret_cast<const bf16x8*>(&sa[cb][3][o]);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        accr[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahr, bh[c], accr[r][c], 0, 0, 0);
        acci[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi, bh[c], acci[r][c], 0, 0, 0);
        accr[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahr, bl[c], accr[r][c], 0, 0, 0);
        acci[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ahi, bl[c], acci[r][c], 0, 0, 0);
        accr[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(alr, bh[c], accr[r][c], 0, 0, 0);
        acci[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ali, bh[c], acci[r][c], 0, 0, 0);
      }
    }
    // step ks+1 into the other buffer (its readers finished at the last
    // barrier), step ks+2 in flight, then one barrier
    if (ks + 1 < nk) {
      store_c(cb ^ 1);
      if (ks + 2 < nk) load_c(k0 + 2 * kGK);
    }
    __syncthreads();
  }
  // f32 MFMA layout: item i of lane l is row 4*(l/16)+i, column l%16
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t a = a0 + wa + 16 * r + 4 * (lane >> 4) + i;
        const int64_t b = b0 + wb + 16 * c + (lane & 15);
        if (a < lena && b < lenb) {
          float2* d = reinterpret_cast<float2*>(out + (a * lenb + b) * 2);
          *d = make_float2(accr[r][c][i], acci[r][c][i]);
        }
      }
}

// FP64 GEMM tile: 128 rows (alpha strings) x 128 columns (target beta
// strings) per workgroup of 8 waves in a 4 x 2 arrangement, 32 x 64 per
// wave (2 x 4 MFMA tiles, real and imaginary accumulators), K (source beta
// strings) in steps of 16.  Both operands are staged through LDS: the C
// tile as separate real / imaginary planes [k][row] (the A operand), the
// Hbb columns as [k][col] (the B operand, hcol[Ib][Ib'] = Hbb[Ib'][Ib] is
// already K-major).  The next K step's global loads are in flight during
// the MFMAs of the current one.
constexpr int kFK = 16;                   // K step
constexpr int kFS = kGT + 16;             // doubles per LDS row (padding)

__global__ void __launch_bounds__(512, 1)
k_beta_gemm_f64(int64_t lena, int64_t lenb, const double* __restrict__ hcol,
                const double* __restrict__ coeff, double* __restrict__ out,
                const int32_t* __restrict__ done, int ta, int tb,
                int per_xcd) {
  // two buffers of each tile: the next K step is stored while the current
  // one feeds the MFMAs (one barrier per step)
  __shared__ __align__(16) double cre[2][kFK * kFS];
  __shared__ __align__(16) double cim[2][kFK * kFS];
  __shared__ __align__(16) double hb[2][kFK * kFS];
  if (done && *done) return;
  int tile_a, tile_b;
  if (!xcd_tile(ta, tb, per_xcd, &tile_a, &tile_b)) return;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int64_t a0 = static_cast<int64_t>(tile_a) * kGT;
  const int64_t b0 = static_cast<int64_t>(tile_b) * kGT;
  const int wa = (wave >> 1) * 32;        // wave row offset in the tile
  const int wb = (wave & 1) * 64;         // wave column offset
  const __amdgpu_buffer_rsrc_t rc = rsrc(coeff, lena * lenb * 2 * sizeof(double));
  const __amdgpu_buffer_rsrc_t rh = rsrc(hcol, lenb * lenb * sizeof(double));

  // C loader: thread -> tile row tid/4, complex k 4*(tid%4)..+3
  const int cr = tid >> 2;
  const int ck = 4 * (tid & 3);
  const int64_t arow = a0 + cr;
  const bool rowok = arow < lena;
  // Hbb loader: thread -> k row tid/32, columns 4*(tid%32)..+3
  const int hk = tid >> 5;
  const int hn = 4 * (tid & 31);
  u32x4 cv[4];
  uint64_t hv[4];
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t k = k0 + ck + j;
      const int off = (rowok && k < lenb)
                          ? static_cast<int>((arow * lenb + k) * 2 * sizeof(double)) : -1;
      cv[j] = __builtin_amdgcn_raw_buffer_load_b128(rc, off, 0, 0);
    }
    const int64_t k = k0 + hk;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int64_t n = b0 + hn + j;
      const int off = (k < lenb && n < lenb)
                          ? static_cast<int>((k * lenb + n) * sizeof(double)) : -1;
      const u32x2 y = __builtin_amdgcn_raw_buffer_load_b64(rh, off, 0, 0);
      hv[j] = static_cast<uint64_t>(y[0]) | (static_cast<uint64_t>(y[1]) << 32);
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint64_t re = static_cast<uint64_t>(cv[j][0]) | (static_cast<uint64_t>(cv[j][1]) << 32);
      const uint64_t im = static_cast<uint64_t>(cv[j][2]) | (static_cast<uint64_t>(cv[j][3]) << 32);
      cre[buf][(ck + j) * kFS + cr] = __longlong_as_double(static_cast<long long>(re));
      cim[buf][(ck + j) * kFS + cr] = __longlong_as_double(static_cast<long long>(im));
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      hb[buf][hk * kFS + hn + j] = __longlong_as_double(static_cast<long long>(hv[j]));
  };

  double4_t accr[2][4], acci[2][4];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      accr[r][c] = double4_t{0, 0, 0, 0};
      acci[r][c] = double4_t{0, 0, 0, 0};
    }

  const int64_t nk = (lenb + kFK - 1) / kFK;
  load(0);
  store(0);
  if (nk > 1) load(kFK);                  // step 1 in flight
  __syncthreads();
  for (int64_t ks = 0; ks < nk; ++ks) {
    const int cb = static_cast<int>(ks & 1);
    // f64 MFMA operands: A[r = l%16][k = l/16], B[k = l/16][c = l%16]
#pragma unroll
    for (int kq = 0; kq < kFK / 4; ++kq) {
      const int krow = (4 * kq + (lane >> 4)) * kFS;
      double ar[2], ai[2], bv[4];
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        ar[r] = cre[cb][krow + wa + 16 * r + (lane & 15)];
        ai[r] = cim[cb][krow + wa + 16 * r + (lane & 15)];
      }
#pragma unroll
      for (int c = 0; c < 4; ++c) bv[c] = hb[cb][krow + wb + 16 * c + (lane & 15)];
#pragma unroll
      for (int r = 0; r < 2; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          accr[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ar[r], bv[c], accr[r][c], 0, 0, 0);
          acci[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ai[r], bv[c], acci[r][c], 0, 0, 0);
        }
    }
    // step ks+1 into the other buffer (its readers finished at the last
    // barrier), step ks+2 in flight, then one barrier
    if (ks + 1 < nk) {
      store(cb ^ 1);
      if (ks + 2 < nk) load((ks + 2) * kFK);
    }
    __syncthreads();
  }
  // f64 MFMA layout: item i of lane l is row l/16 + 4 i, column l%16
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int64_t a = a0 + wa + 16 * r + (lane >> 4) + 4 * i;
        const int64_t b = b0 + wb + 16 * c + (lane & 15);
        if (a < lena && b < lenb) {
          double2* d = reinterpret_cast<double2*>(out + (a * lenb + b) * 2);
          *d = make_double2(accr[r][c][i], acci[r][c][i]);
        }
      }
}

}  // namespace

bool beta_gemm_f64_shape_ok(int64_t lena, int64_t lenb) {
  const int64_t lim = int64_t(1) << 31;
  return lena * lenb * 2 * static_cast<int64_t>(sizeof(double)) < lim &&
         lenb * lenb * static_cast<int64_t>(sizeof(double)) < lim;
}

int launch_beta_gemm_f64(int64_t lena, int64_t lenb, const double* hcol,
                         const double* coeff, double* out, hipStream_t st,
                         const int32_t* done) {
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  const int ta = static_cast<int>((lena + kGT - 1) / kGT);
  const int tb = static_cast<int>((lenb + kGT - 1) / kGT);
  const int per_xcd = (ta * tb + kXcds - 1) / kXcds;
  k_beta_gemm_f64<<<static_cast<unsigned>(per_xcd * kXcds), 512, 0, st>>>(
      lena, lenb, hcol, coeff, out, done, ta, tb, per_xcd);
  FQEHIP_CHECK_LAUNCH("k_beta_gemm_f64");
  return FQEHIP_OK;
}

bool beta_gemm_shape_ok(int64_t lena, int64_t lenb, int64_t ldh) {
  const int64_t lim = int64_t(1) << 31;
  return ldh >= lenb && ldh % kGT == 0 && ldh * ldh * 2 < lim &&
         lena * lenb * 2 * static_cast<int64_t>(sizeof(float)) < lim;
}

int launch_beta_gemm(int64_t lena, int64_t lenb, int64_t ldh, const void* hhi,
                     const void* hlo, const float* coeff, float* out,
                     hipStream_t st, const int32_t* done) {
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  const int ta = static_cast<int>((lena + kGT - 1) / kGT);
  const int tb = static_cast<int>((lenb + kGT - 1) / kGT);
  const int per_xcd = (ta * tb + kXcds - 1) / kXcds;
  k_beta_gemm_bf16x3<<<static_cast<unsigned>(per_xcd * kXcds), 256, 0, st>>>(
      lena, lenb, ldh, static_cast<const __bf16*>(hhi),
      static_cast<const __bf16*>(hlo), coeff, out, done, ta, tb, per_xcd);
  FQEHIP_CHECK_LAUNCH("k_beta_gemm_bf16x3");
  return FQEHIP_OK;
}

}  // namespace fqehip

using namespace fqehip;

extern "C" int64_t fqehip_beta_block_ld(int64_t lenb) {
  return lenb <= 0 ? 0 : ((lenb + kGT - 1) / kGT) * kGT;
}

extern "C" int fqehip_beta_block(int npair, int64_t lenb, const int32_t* d_fwd_b,
                                 const double* d_a, double* d_hcol,
                                 uint16_t* d_hhi, uint16_t* d_hlo, int64_t ldh,
                                 void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(npair >= 0 && lenb >= 0, "npair=%d lenb=%lld", npair,
                   static_cast<long long>(lenb));
  FQEHIP_CHECK_ARG(ldh == fqehip_beta_block_ld(lenb),
                   "ldh=%lld, expected %lld", static_cast<long long>(ldh),
                   static_cast<long long>(fqehip_beta_block_ld(lenb)));
  FQEHIP_CHECK_ARG((lenb + npair) * static_cast<int64_t>(sizeof(double)) <= 160 * 1024,
                   "lenb=%lld exceeds the LDS column of the beta block",
                   static_cast<long long>(lenb));
  if (lenb == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_a && d_hcol && d_hhi && d_hlo, "NULL pointer");
  FQEHIP_CHECK_ARG(npair == 0 || d_fwd_b, "NULL beta forward table");
  hipStream_t st = as_stream(stream);
  int rc = spin_block<false>(npair, lenb, d_fwd_b, d_a, npair,
                             d_a + static_cast<int64_t>(npair) * npair, d_hcol, st);
  if (rc) return rc;
  dim3 grid(static_cast<unsigned>(ldh / 32), static_cast<unsigned>(ldh / 32));
  k_beta_split<<<grid, 256, 0, st>>>(lenb, ldh, d_hcol,
                                      reinterpret_cast<__bf16*>(d_hhi),
                                      reinterpret_cast<__bf16*>(d_hlo));
  FQEHIP_CHECK_LAUNCH("k_beta_split");
  return FQEHIP_OK;
}

extern "C" int fqehip_spin_block(int complex_op, int npair, int64_t len,
                                 const int32_t* d_fwd, const double* d_v,
                                 int64_t lda, const double* d_h, double* d_hcol,
                                 void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(complex_op == 0 || complex_op == 1, "complex_op=%d", complex_op);
  const int64_t w = complex_op ? 2 : 1;
  FQEHIP_CHECK_ARG(npair >= 0 && len >= 0 && lda >= w * npair,
                   "npair=%d len=%lld lda=%lld", npair,
                   static_cast<long long>(len), static_cast<long long>(lda));
  const size_t lds = static_cast<size_t>(len + npair) * sizeof(double) * w;
  FQEHIP_CHECK_ARG(lds <= 160 * 1024, "len=%lld exceeds the LDS column of the block",
                   static_cast<long long>(len));
  if (len == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_hcol && (npair == 0 || (d_fwd && d_v && d_h)), "NULL pointer");
  hipStream_t st = as_stream(stream);
  return complex_op ? spin_block<true>(npair, len, d_fwd, d_v, lda, d_h, d_hcol, st)
                    : spin_block<false>(npair, len, d_fwd, d_v, lda, d_h, d_hcol, st);
}

extern "C" int fqehip_beta_gemm(int64_t lena, int64_t lenb,
                                const uint16_t* d_hhi, const uint16_t* d_hlo,
                                int64_t ldh, const void* d_coeff, void* d_out,
                                const int32_t* d_done, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(lena >= 0 && lenb >= 0, "negative size");
  FQEHIP_CHECK_ARG(beta_gemm_shape_ok(lena, lenb, ldh),
                   "ldh=%lld does not fit lenb=%lld (multiple of %d needed)",
                   static_cast<long long>(ldh), static_cast<long long>(lenb), kGT);
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_hhi && d_hlo && d_coeff && d_out, "NULL pointer");
  return launch_beta_gemm(lena, lenb, ldh, d_hhi, d_hlo,
                          static_cast<const float*>(d_coeff),
                          static_cast<float*>(d_out), as_stream(stream), d_done);
}

extern "C" int fqehip_beta_gemm_f64(int64_t lena, int64_t lenb,
                                    const double* d_hcol, const void* d_coeff,
                                    void* d_out, const int32_t* d_done,
                                    void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(lena >= 0 && lenb >= 0, "negative size");
  FQEHIP_CHECK_ARG(beta_gemm_f64_shape_ok(lena, lenb),
                   "lena=%lld lenb=%lld too large for 32-bit offsets",
                   static_cast<long long>(lena), static_cast<long long>(lenb));
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_hcol && d_coeff && d_out, "NULL pointer");
  return launch_beta_gemm_f64(lena, lenb, d_hcol,
                              static_cast<const double*>(d_coeff),
                              static_cast<double*>(d_out), as_stream(stream),
                              d_done);
}
