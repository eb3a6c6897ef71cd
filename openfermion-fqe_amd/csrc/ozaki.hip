// Ozaki-digit variant of the pull form (pull.hip) for complex128 applies of
// pair-symmetric real operators: the same operands and the same three parts
// H C = Haa C + C Hbb^T + sum_q E^b_q (sum_p W[p][q] E^a_p C), with every
// product formed exactly from 8-bit digits on the matrix cores
// (v_mfma_i32_16x16x64_i8, int32 accumulation) instead of FP64 matrix-core
// products, and assembled in FP64.
//
// Digits.  An operator row (of W: all alpha pairs p of one beta pair q; of
// Haa, Hbb: all source strings of one target) is scaled by a power of two so
// that |x 2^ea| < 2^38, rounded to the integer z and split exactly into five
// balanced signed digits a_0..a_4 in [-128, 127] of weights 2^32, 2^24, ..., 1
// (from the low end: d = ((z + 128) mod 256) - 128, z = (z - d) / 256).
// Data (C) is scaled by one power of two per alpha string (rows and Hbb) or
// beta string (Haa), from a bound on the magnitudes, so that |x 2^ed| < 2^46,
// and rounded to a 48-bit integer y.  The six bytes of y (two's complement)
// are the digits d_0..d_5 of weights 1 .. 2^40.  d_0..d_4 are stored as
// unsigned bytes minus 128 (one XOR), d_5 as the signed top byte, so no carry
// propagation is needed; the 128 offsets are added back exactly, for every
// digit pair, through the sums of the operator integers.  Data that are all zero
// have no scale and get a zero factor on the way back: the offsets of the
// digit pairs that are not formed (below) would be left in the result.
//
// Products.  Of the 30 digit pairs, the 20 with i - t >= 0 (weight >= 2^32
// of a maximum of 2^72) are formed, six int32 accumulators per output (one
// per i - t); the dropped pairs weigh at most 2^-40 of the largest product
// each, and since the offsets of all pairs are corrected, they enter as
// sums of zero-mean terms: about 1e-11 of the result when the bound is a
// few times the values, and still below 1e-9 for vectors whose weight sits
// on a few determinants.  Every int32 sum is exact.  A result is assembled in
// FP64: 2^-(ea+ed) (2^32 sum_m 2^(8m) acc_m + 128 (1 + 2^8 + 2^16 + 2^24 +
// 2^32) sum z).
//
// Reference: lm_apply_array12_same_spin_opt / lm_apply_array12_diff_spin_opt
// (src/fqe/lib/fqe_data.c:668-720, :879-996), in complex128.
#include <type_traits>

#include "fqehip_common.h"
#include "pull_common.h"
#include "rows_common.h"

namespace fqehip {
namespace {

using namespace rows;

typedef int int4v __attribute__((ext_vector_type(4)));

constexpr int kOzK = 64;                   // live alpha pairs of a string, padded
constexpr int kOzADig = 5;                 // digits of the operator
constexpr int kOzDDig = 6;                 // digits 0..5 of the data integers
constexpr int kOzARow = kOzK + 16;         // bytes per LDS row of a digit plane
constexpr int kOzQ = 128;                  // beta pairs, padded (table pitch)
constexpr double kMagic = 6755399441055744.0;  // 1.5 * 2^52: rint via one add

// max(m, |v|), infinity from a NaN on
__device__ __forceinline__ double absmax(double m, double v) {
  return v == v ? fmax(m, fabs(v)) : HUGE_VAL;
}

// 2^-e, the factor back of data with the maximum m scaled by 2^e: zero where all
// are zero, and NaN where one is not finite and has no digits.
__device__ __forceinline__ double factor_back(double m, int e) {
  return m > 0.0 ? (m < HUGE_VAL ? ldexp(1.0, -e) : __longlong_as_double(0x7ff8000000000000ll)) : 0.0;
}

// rowmax[I] = max over the row of max(|Re C[I][.]|, |Im C[I][.]|), infinity where
// one is not finite; zeroes colmax (when not NULL) for k_col_absmax and the nsum
// sums of k_pull_rows_oz.
__global__ void __launch_bounds__(256)
k_row_absmax(int64_t lena, int64_t lenb, const double* __restrict__ coeff,
             double* __restrict__ rowmax, unsigned long long* __restrict__ colmax,
             unsigned long long* __restrict__ sums, int64_t nsum,
             const int32_t* __restrict__ done) {
  __shared__ double red[4];
  if (done && *done) return;
  if (colmax)
    for (int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; j < lenb;
         j += static_cast<int64_t>(gridDim.x) * 256)
      colmax[j] = 0;
  for (int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x; j < nsum;
       j += static_cast<int64_t>(gridDim.x) * 256)
    sums[j] = 0;
  for (int64_t r = blockIdx.x; r < lena; r += gridDim.x) {
    const double* row = coeff + r * lenb * 2;
    double m = 0.0;
    for (int64_t k = threadIdx.x; k < 2 * lenb; k += 256) m = absmax(m, row[k]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0)
      rowmax[r] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    __syncthreads();
  }
}

// colmax[j] = the same over column j (bits of a non-negative double, ordered
// as the doubles are), 64 rows per workgroup.
constexpr int kColRows = 64;
__global__ void __launch_bounds__(256)
k_col_absmax(int64_t lena, int64_t lenb, const double* __restrict__ coeff,
             unsigned long long* __restrict__ colmax,
             const int32_t* __restrict__ done) {
  if (done && *done) return;
  const int64_t j = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (j >= lenb) return;
  const int64_t r0 = static_cast<int64_t>(blockIdx.y) * kColRows;
  const int64_t r1 = r0 + kColRows < lena ? r0 + kColRows : lena;
  double m = 0.0;
#pragma unroll 8
  for (int64_t r = r0; r < r1; ++r) {
    const double2 v = reinterpret_cast<const double2*>(coeff)[r * lenb + j];
    m = absmax(absmax(m, v.x), v.y);
  }
  atomicMax(&colmax[j], static_cast<unsigned long long>(__double_as_longlong(m)));
}

// Digits 0..5 of four 48-bit integers y_j held as the (lo, hi) words of
// kMagic + y_j: out[i] byte j = digit i of y_j (bytes 0..3 of lo, bytes 0..1
// of hi); digits 0..4 are unsigned bytes offset by -128 (one XOR), digit 5
// is the signed top byte.  A two-stage byte transpose with v_perm_b32
// (perm(a, b, sel): result byte k = byte sel_k of the 8 bytes b0..b3 a0..a3).
__device__ __forceinline__ void digits_of_four(const uint32_t (&lo)[4],
                                               const uint32_t (&hi)[4],
                                               uint32_t (&out)[6]) {
  // x01 = [lo0.b0, lo1.b0, lo0.b1, lo1.b1], y01 = [lo0.b2, lo1.b2, lo0.b3, lo1.b3]
  const uint32_t x01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x05010400u);
  const uint32_t y01 = __builtin_amdgcn_perm(lo[1], lo[0], 0x07030602u);
  const uint32_t x23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x05010400u);
  const uint32_t y23 = __builtin_amdgcn_perm(lo[3], lo[2], 0x07030602u);
  const uint32_t z01 = __builtin_amdgcn_perm(hi[1], hi[0], 0x05010400u);
  const uint32_t z23 = __builtin_amdgcn_perm(hi[3], hi[2], 0x05010400u);
  out[0] = __builtin_amdgcn_perm(x23, x01, 0x05040100u) ^ 0x80808080u;
  out[1] = __builtin_amdgcn_perm(x23, x01, 0x07060302u) ^ 0x80808080u;
  out[2] = __builtin_amdgcn_perm(y23, y01, 0x05040100u) ^ 0x80808080u;
  out[3] = __builtin_amdgcn_perm(y23, y01, 0x07060302u) ^ 0x80808080u;
  out[4] = __builtin_amdgcn_perm(z23, z01, 0x05040100u) ^ 0x80808080u;
  out[5] = __builtin_amdgcn_perm(z23, z01, 0x07060302u);
}

__device__ __forceinline__ void split_words(double v, uint32_t& lo,
                                            uint32_t& hi) {
  const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
  lo = static_cast<uint32_t>(b);
  hi = static_cast<uint32_t>(b >> 32);
}

__device__ __forceinline__ double as_double(uint32_t lo, uint32_t hi) {
  return __longlong_as_double(static_cast<long long>(
      static_cast<uint64_t>(lo) | (static_cast<uint64_t>(hi) << 32)));
}

// Offset correction constant: the -128 offsets of data digits 0..4 over
// every digit pair, 128 (1 + 2^8 + 2^16 + 2^24 + 2^32) per unit of the
// operator integers' sum.
constexpr double kOffsetUnit = 128.0 * 4311810305.0;
// Invalid row offset, in 16-byte units: (kNoRow16 + column) * 16 lies past the
// end of C (lena * lenb * 16 <= 0x7ff00000 is a launch requirement) and below
// 2^31 (lenb < 2^16).
constexpr uint32_t kNoRow16 = 0x7ff0000u;

// Tables of W for the row kernel, once per operator: the digits of every
// alpha pair's column, dig[p][t][q] bytes (t: digit of weight 2^(8(4 - t))),
// the integers z[p][q] = rint(W 2^ea[q]) as doubles, |z| < 2^38, each row q with
// the scale of its own largest element; the exponent e of the accumulators'
// unit 2^(32 - e) (in units of the data), one for all of W: sum_pq |W| 2^e <
// 2^49, so that a sum over any (p, q) of W 2^e times 46-bit data, in units of
// 2^32, stays below 2^63; and what takes a row's products to that unit, shifts
// to the right by ea[q] - e as bytes.  Without left shifts e is at most the
// smallest ea, which is as fine as the digits of rows down to 2^-12 of the
// largest one (the sums' rounding, a few units, is then 2^-49 of the largest
// row, theirs 2^-38 of their own); beside a row that is smaller still, e is 12
// below that row's ea, or at the limit of the sum, and the left_rows rows above
// it shift to the left.
// ea[q] is held to e + 31, where a whole row's digits are finer than the unit.  One
// workgroup per pair p, thread q; every workgroup forms the maximum and the
// sum anew, in one order.
struct OzUnit {
  int32_t e;
  uint32_t left_rows;
  uint8_t right[kOzQ], left[kOzQ];
};
constexpr int64_t kWDigBytes = static_cast<int64_t>(kOzADig) * kOzQ;
__global__ void __launch_bounds__(kOzQ)
k_pull_digits(int npull, const double* __restrict__ w, uint8_t* __restrict__ dig,
              double* __restrict__ z, OzUnit* __restrict__ unit) {
  __shared__ double red[2][kOzQ / 64];
  __shared__ uint32_t rows;
  __shared__ int least[kOzQ / 64];
  const int p = blockIdx.x;
  const int q = threadIdx.x;
  double m = 0.0, t = 0.0;
  if (q < npull) {
#pragma unroll 8
    for (int r = 0; r < npull; ++r) {
      const double v = fabs(w[static_cast<int64_t>(r) * npull + q]);
      m = fmax(m, v);
      t += v;
    }
  }
  const double mq = m;
  int emin = 4096;                         // exponent of the smallest row
  if (mq > 0.0) (void)frexp(mq, &emin);
  if (q == 0) rows = 0;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    m = fmax(m, __shfl_xor(m, o));
    t += __shfl_xor(t, o);
    const int x = __shfl_xor(emin, o);
    emin = x < emin ? x : emin;
  }
  if ((q & 63) == 0) {
    red[0][q >> 6] = m;
    red[1][q >> 6] = t;
    least[q >> 6] = emin;
  }
  __syncthreads();
  emin = least[0] < least[1] ? least[0] : least[1];
  m = fmax(red[0][0], red[0][1]);
  t = red[1][0] + red[1][1];
  int e = 0, eq = 0;
  if (m > 0.0) {
    int em, et;
    (void)frexp(m, &em);
    (void)frexp(t * (1.0 + 0x1p-20), &et);   // the z are rounded
    e = em - emin > 12 ? 26 - emin : 38 - em;
    e = e < 49 - et ? e : 49 - et;
    eq = e;
    if (mq > 0.0) {
      (void)frexp(mq, &em);
      eq = 38 - em < e + 31 ? 38 - em : e + 31;
    }
  }
  int64_t v = q < npull ? static_cast<int64_t>(rint(ldexp(w[static_cast<int64_t>(p) * npull + q], eq))) : 0;
  z[static_cast<int64_t>(p) * kOzQ + q] = static_cast<double>(v);
  if (p == 0) {
    if (eq < e) atomicAdd(&rows, 1u);
    unit->right[q] = static_cast<uint8_t>(eq > e ? eq - e : 0);
    unit->left[q] = static_cast<uint8_t>(eq < e ? e - eq : 0);
    __syncthreads();                       // p is the workgroup's
    if (q == 0) {
      unit->e = e;
      unit->left_rows = rows;
    }
  }
#pragma unroll
  for (int t5 = kOzADig - 1; t5 >= 0; --t5) {
    const int64_t d = t5 ? ((v + 128) & 255) - 128 : v;
    v = (v - d) >> 8;
    dig[p * kWDigBytes + t5 * kOzQ + q] = static_cast<uint8_t>(d & 0xff);
  }
}

// Opposite-spin rows, one alpha string ia per workgroup of 8 waves (see
// k_pull_rows_f64 for the operands).  K is the de-excitation rows of ia as
// they are, diagonal ones included: at most 64, one k step of the i8 MFMA.
//
// Set-up: row offsets, signs and the scale of the data; the digits of the
// live columns of W transposed from dig[p][t][q] to [t][q][k] in LDS, four k
// by four q at a time (v_perm_b32); and per q the offset correction from the
// sum of the integers, split into the three int32 start values of the
// accumulator classes 0, 2 and 4.
//
// Main loop: each wave owns 16 columns of a 128-column chunk, loads its C
// values (lane l: column l%16, k = 16 (l/16) + j) two batches of four ahead,
// forms the six digit operands in registers, and runs the 20 digit products
// of every 16-row tile of W for the real and the imaginary part on the same
// A operands.  i8 MFMA layouts: lane l holds A[row l%16][k 16 (l/16) + j] and
// B[k 16 (l/16) + j][col l%16]; output item e is [row 4 (l/16) + e][col l%16].
//
// A value is the 64-bit integer sum_m 2^(8m) acc_m in its row's unit
// 2^(32 - ea[q] - ed), assembled with 32-bit integer operations and shifted
// to the accumulators' unit 2^(32 - e - ed); it is added to its target's
// 64-bit accumulator in LDS (ds_add_u64).  Integer addition has no order, so the
// waves need no turns and every run gives the same bits.  The shift rounds down
// and a negative sign of E^b_q is one XOR (-v - 1), half a unit low on average
// each way, so the accumulators start at half a unit for each excitation that
// reaches them; what is left is a few units.  The shift keeps the digits of a row
// as fine as its own largest element allows (one scale for all of W would round
// every row as the largest one, 0 to 3 bits for integrals of canonical orbitals,
// and the whole ratio beside one large local integral).  norb 14 7a7b: 3.1 ms,
// with the shift and, signed halves extended instead, without it; 3.7 with FP64
// assembly (four v_cvt_f64_i32 per value);
// without the products 2.4, without the additions 2.4, set-up alone 0.24 (the
// slot-row form of the same products: 4.0 + 1.3 for its reduction).  Two waves
// per SIMD fit (256 registers), so products and additions overlap only in part.
struct OzRowsArgs {
  int norb, compressed, nalpha, nq, nqt;
  int64_t lena, lenb;
  const uint8_t* dig;
  const double* z;
  const OzUnit* unit;
  const int32_t* dexc;
  int half;                                // accumulators' start value
  const uint32_t* fwd;
  const double* coeff;
  const double* rowmax;
  double* rowacc;
  double alpha_re, alpha_im, beta_re, beta_im;
  const double* cin;
  double* out;
  double* acc;
  double* partials;
  const int32_t* done;
  int nseg;                                // workgroups per alpha string
  unsigned long long* sums;                // nseg > 1: [lena][lenb][re, im]
  double* back;                            // and each row's factor
};

constexpr int kRowThreads = 512;
constexpr int kRowCols = 128;              // columns per chunk of 8 waves
constexpr int kOzPartBytes = 4 * kOzQ * 8;   // set-up scratch

size_t oz_rows_lds_bytes(int64_t lenb, int nqt) {
  const size_t acc = static_cast<size_t>(lenb) * 16;
  return (acc > kOzPartBytes ? acc : kOzPartBytes) +
         static_cast<size_t>(kOzADig) * 16 * nqt * kOzARow + 3 * kOzQ * 4 + 2 * kOzQ +
         kOzK * (8 + 4 + 4) + 16;
}

// The finished row ia: rowacc + back * value(x), and the epilogue.
template <typename F>
__device__ __forceinline__ void oz_finish(const OzRowsArgs& p, int64_t ia, double back,
                                          F value, char* smem) {
  double2* racc = reinterpret_cast<double2*>(p.rowacc) + ia * p.lenb;
  double sq = 0.0;
  for (int x = threadIdx.x; x < static_cast<int>(p.lenb); x += kRowThreads) {
    const double2 r = racc[x];
    const double re = r.x + back * static_cast<double>(static_cast<int64_t>(value(2 * x)));
    const double im = r.y + back * static_cast<double>(static_cast<int64_t>(value(2 * x + 1)));
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
      p.acc[2 * idx] += vr;
      p.acc[2 * idx + 1] += vi;
    }
  }
  if (p.partials) row_norm(sq, p.partials + ia, smem);
}

__global__ void __launch_bounds__(kRowThreads, 2) k_pull_rows_oz(OzRowsArgs p) {
  extern __shared__ __align__(16) char smem[];
  if (p.done && *p.done) return;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int kq = lane >> 4;
  const int cl = lane & 15;
  const int lenb = static_cast<int>(p.lenb);
  const int nqp = 16 * p.nqt;
  // nseg workgroups share a row, each with its part of the column chunks
  const int64_t ia = p.nseg > 1 ? blockIdx.x / p.nseg : xcd_order(blockIdx.x, p.lena);
  const int seg = p.nseg > 1 ? static_cast<int>(blockIdx.x) % p.nseg : 0;
  const int accb = lenb * 16 > kOzPartBytes ? lenb * 16 : kOzPartBytes;
  unsigned long long* accs = reinterpret_cast<unsigned long long*>(smem);  // [lenb][re, im]
  double* part = reinterpret_cast<double*>(smem);       // set-up: [4][kOzQ]
  uint8_t* adig = reinterpret_cast<uint8_t*>(smem + accb);   // [5][nqp][kOzARow]
  int32_t* start = reinterpret_cast<int32_t*>(adig + kOzADig * nqp * kOzARow);  // [3][kOzQ]
  uint32_t* shift = reinterpret_cast<uint32_t*>(start + 3 * kOzQ);   // right, left: bytes
  double* gsa = reinterpret_cast<double*>(shift + kOzQ / 2);  // [kOzK] sign 2^ed
  uint32_t* goff = reinterpret_cast<uint32_t*>(gsa + kOzK);
  int32_t* lp = reinterpret_cast<int32_t*>(goff + kOzK);
  double* scale = reinterpret_cast<double*>(lp + kOzK);  // 2^-ed
  const int nexc = p.nalpha * (p.norb - p.nalpha + 1);

  if (wave == 0) {
    int32_t src = 0, ij = 0, sg = 0;
    double m = 0.0;
    if (lane < nexc) {
      const int32_t* e = p.dexc + (ia * nexc + lane) * 3;
      src = e[0];
      ij = e[1];
      sg = e[2];
      m = p.rowmax[src];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o));
    int e = 0;
    if (m > 0.0) {
      (void)frexp(m, &e);
      e = 46 - e;                           // |D 2^ed| < 2^46
    }
    const int i = ij / p.norb, j = ij % p.norb;
    lp[lane] = lane < nexc ? (p.compressed ? comp_pair(i, j) : ij) : -1;
    goff[lane] = lane < nexc ? static_cast<uint32_t>(src) * static_cast<uint32_t>(lenb) : kNoRow16;
    gsa[lane] = static_cast<double>(sg) * ldexp(1.0, e);
    if (lane == 0) *scale = factor_back(m, e);
  }
  __syncthreads();
  {
    const int q = tid & (kOzQ - 1);
    const int k0 = (tid >> 7) * 16;
    double zs = 0.0;
#pragma unroll
    for (int k = k0; k < k0 + 16; ++k) zs += k < nexc ? p.z[lp[k] * kOzQ + q] : 0.0;
    part[(tid >> 7) * kOzQ + q] = zs;
  }
  // W digits: block x = (t, four q, four k)
  for (int x = tid; x < kOzADig * (nqp / 4) * (kOzK / 4); x += kRowThreads) {
    const int k4 = x & 15;
    const int tq = x >> 4;
    const int t = tq / (nqp / 4);
    const int q4 = tq - t * (nqp / 4);
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int pr = lp[4 * k4 + u];
      v[u] = pr >= 0 ? *reinterpret_cast<const uint32_t*>(p.dig + pr * kWDigBytes + t * kOzQ + 4 * q4)
                     : 0u;
    }
    // transpose: word y holds bytes (q 4 q4 + y) of k 4 k4 .. + 3
    const uint32_t x01 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u);
    const uint32_t y01 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u);
    const uint32_t x23 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u);
    const uint32_t y23 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
    uint8_t* dst = adig + (t * nqp + 4 * q4) * kOzARow + 4 * k4;
    *reinterpret_cast<uint32_t*>(dst) = __builtin_amdgcn_perm(x23, x01, 0x05040100u);
    *reinterpret_cast<uint32_t*>(dst + kOzARow) = __builtin_amdgcn_perm(x23, x01, 0x07060302u);
    *reinterpret_cast<uint32_t*>(dst + 2 * kOzARow) = __builtin_amdgcn_perm(y23, y01, 0x05040100u);
    *reinterpret_cast<uint32_t*>(dst + 3 * kOzARow) = __builtin_amdgcn_perm(y23, y01, 0x07060302u);
  }
  __syncthreads();
  if (tid < kOzQ) {
    // 128 (1 + 2^8 + 2^16 + 2^24 + 2^32) sum z in units of 2^32
    const double zs = part[tid] + part[kOzQ + tid] + part[2 * kOzQ + tid] + part[3 * kOzQ + tid];
    const int64_t v = static_cast<int64_t>(rint(kOffsetUnit * 0x1p-32 * zs));
    const int64_t v4 = (v + (int64_t(1) << 31)) >> 32;
    const int64_t r4 = v - (v4 << 32);
    const int64_t v2 = (r4 + (1 << 15)) >> 16;
    // 2^31 + 2^16 (2^31 + 2^15) - 2^32 (2^15 + 1) = 0: so that the first two pairs
    // of classes need no sign extension
    start[tid] = static_cast<int32_t>(r4 - (v2 << 16) + (int64_t(1) << 31));
    start[kOzQ + tid] = static_cast<int32_t>(v2 + (int64_t(1) << 31) + (1 << 15));
    start[2 * kOzQ + tid] = static_cast<int32_t>(v4 - (1 << 15) - 1);
  }
  if (tid < kOzQ / 2) shift[tid] = reinterpret_cast<const uint32_t*>(p.unit->right)[tid];
  __syncthreads();
  for (int x = tid; x < 2 * lenb; x += kRowThreads) accs[x] = seg ? 0 : p.half;
  __syncthreads();

  const __amdgpu_buffer_rsrc_t rc = buffer_of(p.coeff, p.lena * p.lenb * 16);
  const __amdgpu_buffer_rsrc_t rf = buffer_of(p.fwd, static_cast<int64_t>(nqp) * lenb * 4);
  // the target words' offsets are those of element target + 1
  char* accum = smem - 16;
  const int chunks = (lenb + kRowCols - 1) / kRowCols;
  const int first = chunks * seg / p.nseg;
  const int nchunks = chunks * (seg + 1) / p.nseg;
  u32x4 la[3][4];
  auto load = [&](int chunk, int b, u32x4 (&A)[4]) {
    const int jb = chunk * kRowCols + wave * 16 + cl;
    // columns past the row read column 0 and add nothing
    const uint32_t ib = static_cast<uint32_t>(jb < lenb ? jb : 0);
    const uint4 g = *reinterpret_cast<const uint4*>(goff + 16 * kq + 4 * b);
    A[0] = __builtin_amdgcn_raw_buffer_load_b128(rc, static_cast<int>((g.x + ib) << 4), 0, 0);
    A[1] = __builtin_amdgcn_raw_buffer_load_b128(rc, static_cast<int>((g.y + ib) << 4), 0, 0);
    A[2] = __builtin_amdgcn_raw_buffer_load_b128(rc, static_cast<int>((g.z + ib) << 4), 0, 0);
    A[3] = __builtin_amdgcn_raw_buffer_load_b128(rc, static_cast<int>((g.w + ib) << 4), 0, 0);
  };
  // LEFT: some rows shift to the left.  A whole second loop, so that the usual
  // one has no more than its right shifts (as a condition per value 4% slower)
  auto run = [&](auto LEFT) {
  load(first, 0, la[0]);
  load(first, 1, la[1]);
  for (int chunk = first; chunk < nchunks; ++chunk) {
    const int jb = chunk * kRowCols + wave * 16 + cl;
    const bool colok = jb < lenb;
    int4v dd[2][kOzDDig];                   // [re, im][digit]
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (b + 2 < 4) load(chunk, b + 2, la[(b + 2) % 3]);
      uint32_t lre[4], hre[4], lim[4], him[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const u32x4 v = la[b % 3][u];
        const double sa = gsa[16 * kq + 4 * b + u];
        split_words(fma(sa, as_double(v[0], v[1]), kMagic), lre[u], hre[u]);
        split_words(fma(sa, as_double(v[2], v[3]), kMagic), lim[u], him[u]);
      }
      uint32_t ore[kOzDDig], oim[kOzDDig];
      digits_of_four(lre, hre, ore);
      digits_of_four(lim, him, oim);
#pragma unroll
      for (int i = 0; i < kOzDDig; ++i) {
        // the digit words exist here, before the next batch's loads
        asm volatile("" : "+v"(ore[i]), "+v"(oim[i]));
        dd[0][i][b] = static_cast<int>(ore[i]);
        dd[1][i][b] = static_cast<int>(oim[i]);
      }
    }
    // target words of every row tile, ahead of the next chunk's values: loads
    // return in order, so none is waited for behind those
    uint32_t fw[kOzQ / 16][4];
    const int fo = colok ? (4 * kq * lenb + jb) * 4 : -1;
#pragma unroll
    for (int r = 0; r < kOzQ / 16; ++r)
      if (r < p.nqt)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          fw[r][e] = __builtin_amdgcn_raw_buffer_load_b32(
              rf, fo, (16 * r + e) * 4 * lenb, static_cast<int>(0x80000000u));
    if (chunk + 1 < nchunks) {
      load(chunk + 1, 0, la[0]);
      load(chunk + 1, 1, la[1]);
    }
    // the products at a raised wave priority: the SIMD's other wave, loading
    // and converting, issues in the gaps
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int r = 0; r < kOzQ / 16; ++r) {
      if (r >= p.nqt) break;
      int4v a[kOzADig];
#pragma unroll
      for (int t = 0; t < kOzADig; ++t)
        a[t] = *reinterpret_cast<const int4v*>(adig + (t * nqp + 16 * r + cl) * kOzARow + 16 * kq);
      int4v acc[2][6];
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int m = 0; m < 6; ++m)
          acc[c][m] = (m & 1) ? int4v{0, 0, 0, 0}
                              : *reinterpret_cast<const int4v*>(start + (m >> 1) * kOzQ + 16 * r + 4 * kq);
      // pairs (data digit i, operator digit t) with m = i - t >= 0
#pragma unroll
      for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int i = 0; i < kOzDDig; ++i)
#pragma unroll
          for (int t = 0; t < kOzADig; ++t)
            if (t <= i)
              acc[c][i - t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                  a[t], dd[c][i], acc[c][i - t], 0, 0, 0);
      const uint32_t right = shift[4 * r + kq];
      const uint32_t left = LEFT ? shift[kOzQ / 4 + 4 * r + kq] : 0u;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t f = fw[r][e];
        if (!f) continue;
        unsigned long long* to = reinterpret_cast<unsigned long long*>(accum + (f << 1));
        const uint32_t sg = static_cast<uint32_t>(static_cast<int32_t>(f) >> 31);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          // classes merged in pairs in 32 bits: with K <= 64 the odd classes
          // are below 2^22.4 (at most five products of 64 x 2^14), and the
          // first two pairs are positive (see start)
          const uint32_t m10 = static_cast<uint32_t>(acc[c][1][e]) * 256u + acc[c][0][e];
          const uint32_t m32 = static_cast<uint32_t>(acc[c][3][e]) * 256u + acc[c][2][e];
          const uint32_t m54 = static_cast<uint32_t>(acc[c][5][e]) * 256u + acc[c][4][e];
          uint32_t carry, none;
          const uint32_t lo = __builtin_addc(m10, m32 << 16, 0u, &carry);
          const uint32_t hi = __builtin_addc(m54, m32 >> 16, carry, &none);
          int64_t v = static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo);
          if (LEFT) v <<= (left >> (8 * e)) & 63;
          v >>= (right >> (8 * e)) & 63;
          const uint32_t vl = static_cast<uint32_t>(v) ^ sg;
          const uint32_t vh = static_cast<uint32_t>(v >> 32) ^ sg;
          __hip_atomic_fetch_add(to + c, static_cast<unsigned long long>(vh) << 32 | vl,
                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
      }
    }
    __builtin_amdgcn_s_setprio(0);
  }
  };
  if (p.unit->left_rows) run(std::true_type{});
  else run(std::false_type{});
  __syncthreads();
  const double back = ldexp(*scale, 32 - p.unit->e);
  if (p.nseg > 1) {
    unsigned long long* sums = p.sums + ia * p.lenb * 2;
    for (int x = tid; x < 2 * lenb; x += kRowThreads)
      if (accs[x]) atomicAdd(sums + x, accs[x]);
    if (seg == 0 && tid == 0) p.back[ia] = back;
    return;
  }
  oz_finish(p, ia, back, [&](int x) { return accs[x]; }, smem);
}

// The rows that k_pull_rows_oz left as sums over its segments.
__global__ void __launch_bounds__(kRowThreads) k_pull_sums_oz(OzRowsArgs p) {
  __shared__ double red[kRowThreads / 64];
  if (p.done && *p.done) return;
  const int64_t ia = blockIdx.x;
  const unsigned long long* sums = p.sums + ia * p.lenb * 2;
  oz_finish(p, ia, p.back[ia], [&](int x) { return sums[x]; }, reinterpret_cast<char*>(red));
}

constexpr size_t kLdsLimit = 160 * 1024;

}  // namespace

// Whether the digit kernels take a sector of the pull form: at most 64
// de-excitation rows, 128 pairs, the accumulator row in LDS, 32-bit offsets.
bool pull_oz_supported(const fqehip_sector* s) {
  return s->w_oz && s->pull_fwd && s->dexc_a && s->npull <= kOzQ && s->npull > 0 &&
         s->nalpha * (s->norb - s->nalpha + 1) <= kOzK && s->lenb < (1 << 16) &&
         s->lena * s->lenb * 16 <= static_cast<int64_t>(kNoRow16) * 16 &&
         kOzQ * s->lenb * 4 < (int64_t(1) << 31) &&
         oz_rows_lds_bytes(s->lenb, (s->npull + 15) / 16) <= kLdsLimit;
}

// Workgroups per alpha string of the digit rows.  A row is a workgroup until
// there are too few for the chip; then its column chunks are shared out to as
// many as fill it, which are summed in global memory (integers: in any order) at
// the price of a launch and of a set-up each (some 18 us beside 6.5 per chunk).
// Rows of 3432 columns, us with one workgroup / with segments and their sum: 14
// rows 194 / 34, 91 rows 202 / 124; of 6435 columns: 105 rows 409 / 251.
int pull_oz_segments(const fqehip_sector* s) {
  const int64_t fill = 256 / (s->lena > 0 ? s->lena : 1);
  const int64_t chunks = (s->lenb + kRowCols - 1) / kRowCols;
  const int64_t n = fill < chunks ? fill : chunks;
  return n > 1 ? static_cast<int>(n) : 1;
}

// The opposite-spin rows on top of rowacc (epilogue as launch_pull_rows); sums:
// with segments, the zeroed 2 lena lenb integers, then lena doubles.
int launch_pull_rows_oz(const fqehip_sector* s, const double* coeff,
                        const double* rowmax, double* rowacc, double* sums,
                        const PullEpilogue& e, hipStream_t st,
                        const int32_t* done) {
  OzRowsArgs p{};
  p.norb = s->norb;
  p.compressed = s->npull == s->norb * (s->norb + 1) / 2 ? 1 : 0;
  p.nalpha = s->nalpha;
  p.nq = s->npull;
  p.nqt = (s->npull + 15) / 16;
  p.lena = s->lena;
  p.lenb = s->lenb;
  p.dig = static_cast<const uint8_t*>(s->w_oz);
  p.z = reinterpret_cast<const double*>(p.dig + s->npull * kWDigBytes);
  p.unit = reinterpret_cast<const OzUnit*>(p.z + static_cast<int64_t>(s->npull) * kOzQ);
  p.half = s->nbeta * (s->norb - s->nbeta + 1) / 2;
  p.dexc = s->dexc_a;
  p.fwd = s->pull_fwd;
  p.coeff = coeff;
  p.rowmax = rowmax;
  p.rowacc = rowacc;
  p.alpha_re = e.alpha_re;
  p.alpha_im = e.alpha_im;
  p.beta_re = e.beta_re;
  p.beta_im = e.beta_im;
  p.cin = e.cin;
  p.out = e.out;
  p.acc = e.acc;
  p.partials = e.partials;
  p.done = done;
  p.nseg = pull_oz_segments(s);
  p.sums = reinterpret_cast<unsigned long long*>(sums);
  p.back = sums + 2 * s->lena * s->lenb;
  k_pull_rows_oz<<<static_cast<unsigned>(s->lena * p.nseg), kRowThreads,
                   oz_rows_lds_bytes(s->lenb, p.nqt), st>>>(p);
  FQEHIP_CHECK_LAUNCH("k_pull_rows_oz");
  if (p.nseg > 1) {
    k_pull_sums_oz<<<static_cast<unsigned>(s->lena), kRowThreads, 0, st>>>(p);
    FQEHIP_CHECK_LAUNCH("k_pull_sums_oz");
  }
  return FQEHIP_OK;
}

}  // namespace fqehip

// ---------------------------------------------------------------------------
// Same-spin halves: C Hbb^T and Haa C = (C^T Haa^T)^T as digit products on the
// int8 matrix cores, the second on the digits of C^T.
//
//   data: each row of the GEMM's left factor (row Ia of C; row Ib of C^T, i.e.
//      column Ib of C) scaled by 2^ec (|C 2^ec| < 2^46 from its maximum,
//      shared by the real and imaginary parts), rounded to 48-bit integers;
//      digits 0..5 (bytes), 0..4 offset by -128 as in the rows.
//      M index of the GEMM = 2 row + (0 real | 1 imaginary).
//   H: each target's row scaled by 2^eh (|H 2^eh| < 2^38), five balanced
//      digits, built once per operator (fqehip_beta_block_digits) together
//      with the scales and the offset corrections.
// Products with i - t >= 0 (20 pairs), six int32 accumulators per output
// (exact for K < 26214: at most 5 * 128 * 128 * K < 2^31).
// ---------------------------------------------------------------------------
namespace fqehip {
namespace {

constexpr int kBgTM = 128;                  // tile rows (M)
constexpr int kBgTN = 64;                   // tile columns (N)
constexpr int kBgK = 64;                    // K step
constexpr int kBgXcds = 8;                  // XCDs of an MI355X
constexpr int kBgGroup = 8;                 // row tiles per group of the order

// Tile of workgroup blockIdx.x in an order that keeps each XCD on its own
// contiguous run of tiles, grouped kBgGroup row tiles at a time (workgroup
// L runs on XCD L % 8).  False for padding workgroups.
__device__ __forceinline__ bool oz_tile(int tm, int tn, int per_xcd, int* im,
                                        int* in) {
  const int x = static_cast<int>(blockIdx.x % kBgXcds);
  const int t = x * per_xcd + static_cast<int>(blockIdx.x / kBgXcds);
  if (t >= tm * tn) return false;
  const int g = t / (kBgGroup * tn);
  const int left = tm - g * kBgGroup;
  const int rows = left < kBgGroup ? left : kBgGroup;
  const int w = t - g * kBgGroup * tn;
  *im = g * kBgGroup + w % rows;
  *in = w / rows;
  return true;
}

// C digits: thread -> (row Ia, four consecutive columns); rows of ldk
// bytes per (digit, M row); cscale[Ia] = 2^-ec.
__global__ void __launch_bounds__(256)
k_c_digits(int64_t lena, int64_t lenb, int64_t ldk,
           const double* __restrict__ coeff, const double* __restrict__ rowmax,
           uint32_t* __restrict__ cdig, double* __restrict__ cscale,
           const int32_t* __restrict__ done) {
  if (done && *done) return;
  const int64_t groups = ldk / 4;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= lena * groups) return;
  const int64_t ia = idx / groups;
  const int64_t g = idx - ia * groups;
  int ec = 0;
  const double mx = rowmax[ia];
  if (mx > 0.0) {
    int e;
    (void)frexp(mx, &e);
    ec = 46 - e;
  }
  if (g == 0) cscale[ia] = factor_back(mx, ec);
  const double sc = ldexp(1.0, ec);
  uint32_t lre[4], hre[4], lim[4], him[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int64_t k = 4 * g + u;
    double xr = 0.0, xi = 0.0;
    if (k < lenb) {
      const double2 v = reinterpret_cast<const double2*>(coeff)[ia * lenb + k];
      xr = v.x;
      xi = v.y;
    }
    split_words(fma(xr, sc, kMagic), lre[u], hre[u]);
    split_words(fma(xi, sc, kMagic), lim[u], him[u]);
  }
  uint32_t ore[6], oim[6];
  digits_of_four(lre, hre, ore);
  digits_of_four(lim, him, oim);
  const int64_t rows = 2 * lena;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    cdig[((i * rows) + 2 * ia) * groups + g] = ore[i];
    cdig[((i * rows) + 2 * ia + 1) * groups + g] = oim[i];
  }
}

// C^T digits: planes of 2 lenb rows (2 Ib, 2 Ib + 1) of ldk bytes (K = Ia);
// cscale[Ib] = 2^-ec.  A workgroup takes 64 alpha by 32 beta strings: rows of
// C are read coalesced, four consecutive Ia of one column become one word per
// digit, and the words go through LDS to be written 64 bytes per row.
constexpr int kCtA = 64;
constexpr int kCtB = 32;
__global__ void __launch_bounds__(256)
k_ct_digits(int64_t lena, int64_t lenb, int64_t ldk,
            const double* __restrict__ coeff, const double* __restrict__ colmax,
            uint32_t* __restrict__ cdig, double* __restrict__ cscale,
            const int32_t* __restrict__ done) {
  constexpr int kW = kCtA / 4;              // words per row of the tile
  __shared__ uint32_t sm[6][2 * kCtB][kW + 1];
  if (done && *done) return;
  const int64_t b0 = static_cast<int64_t>(blockIdx.x) * kCtB;
  const int64_t a0 = static_cast<int64_t>(blockIdx.y) * kCtA;
  const int jl = threadIdx.x & (kCtB - 1);
  const int64_t jb = b0 + jl;
  int ec = 0;
  const double mx = jb < lenb ? colmax[jb] : 0.0;
  if (mx > 0.0) {
    int e;
    (void)frexp(mx, &e);
    ec = 46 - e;
  }
  if (a0 == 0 && threadIdx.x < kCtB && jb < lenb) cscale[jb] = factor_back(mx, ec);
  const double sc = ldexp(1.0, ec);
  for (int g = threadIdx.x / kCtB; g < kW; g += 256 / kCtB) {
    uint32_t lre[4], hre[4], lim[4], him[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int64_t ia = a0 + 4 * g + u;
      double2 v = make_double2(0.0, 0.0);
      if (ia < lena && jb < lenb) v = reinterpret_cast<const double2*>(coeff)[ia * lenb + jb];
      split_words(fma(v.x, sc, kMagic), lre[u], hre[u]);
      split_words(fma(v.y, sc, kMagic), lim[u], him[u]);
    }
    uint32_t ore[6], oim[6];
    digits_of_four(lre, hre, ore);
    digits_of_four(lim, him, oim);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      sm[i][2 * jl][g] = ore[i];
      sm[i][2 * jl + 1][g] = oim[i];
    }
  }
  __syncthreads();
  const int64_t groups = ldk / 4;
  const int64_t rows = 2 * lenb;
  for (int x = threadIdx.x; x < 6 * 2 * kCtB * kW; x += 256) {
    const int wd = x & (kW - 1);
    const int r = (x / kW) % (2 * kCtB);
    const int i = x / (kW * 2 * kCtB);
    const int64_t row = 2 * b0 + r;
    const int64_t g = a0 / 4 + wd;
    if (row < rows && g < groups) cdig[(i * rows + row) * groups + g] = sm[i][r][wd];
  }
}

// H digits of kHdCols rows Ib' per workgroup (hcol[Ib][Ib']: rows run along
// memory): the row's maximum off the diagonal gives its scale 2^-eh, then five
// exact balanced digits of every K value's integer z, packed four K values
// per word, and the offset correction 128 (1 + 2^8 + 2^16 + 2^24 + 2^32) sum_K z
// (an exact sum of integers, whatever its order).  The diagonal is taken out
// (hdiag, added in FP64 by the GEMM): it is tens of times the other elements
// of its row, and would set the scale they are rounded with (norb 14 7a7b:
// 3.0e-11 normwise with it in the digits).
// A thread takes every kHdK-th word of a row; the words go through LDS so
// that they are written in runs of 256 bytes.  norb 14 (94 MB read twice, 59 MB
// written): 0.19 ms, against 1.15 + 1.70 with a thread per row, 14 workgroups and
// each word of a wave in a line of its own.
constexpr int kHdCols = 16;
constexpr int kHdK = 16;
constexpr int kHdWords = 64;               // words of a row per step

__global__ void __launch_bounds__(kHdCols * kHdK)
k_hbb_digits(int64_t lenb, int64_t ldk, const double* __restrict__ hcol,
             uint32_t* __restrict__ hdig, double* __restrict__ hscale,
             double* __restrict__ hcorr, double* __restrict__ hdiag) {
  __shared__ double red[kHdK][kHdCols];
  __shared__ uint32_t sw[5][kHdCols][kHdWords + 1];
  const int cx = threadIdx.x % kHdCols;
  const int ky = threadIdx.x / kHdCols;
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * kHdCols;
  const int64_t c = c0 + cx;
  const bool ok = c < lenb;
  double m = 0.0;
#pragma unroll 8
  for (int64_t k = ky; k < lenb; k += kHdK) {
    const double v = ok ? fabs(hcol[k * lenb + c]) : 0.0;
    m = fmax(m, k == c ? 0.0 : v);
  }
  red[ky][cx] = m;
  __syncthreads();
  for (int y = 0; y < kHdK; ++y) m = fmax(m, red[y][cx]);
  int eh = 0;
  if (m > 0.0) {
    int e;
    (void)frexp(m, &e);
    eh = 38 - e;
  }
  const int64_t groups = ldk / 4;
  double zsum = 0.0;
  for (int64_t g0 = 0; g0 < groups; g0 += kHdWords) {
#pragma unroll
    for (int j = 0; j < kHdWords / kHdK; ++j) {
      const int64_t g = g0 + ky + kHdK * j;
      uint32_t w[5] = {0u, 0u, 0u, 0u, 0u};
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t k = 4 * g + u;
        const double v = ok && k < lenb && k != c ? hcol[k * lenb + c] : 0.0;
        int64_t z = static_cast<int64_t>(rint(ldexp(v, eh)));
        zsum += static_cast<double>(z);
#pragma unroll
        for (int t = 4; t >= 0; --t) {
          const int64_t d = t ? ((z + 128) & 255) - 128 : z;
          z = (z - d) >> 8;
          w[t] |= (static_cast<uint32_t>(d) & 0xffu) << (8 * u);
        }
      }
#pragma unroll
      for (int t = 0; t < 5; ++t) sw[t][cx][ky + kHdK * j] = w[t];
    }
    __syncthreads();
    for (int x = threadIdx.x; x < 5 * kHdCols * kHdWords; x += kHdCols * kHdK) {
      const int wd = x % kHdWords;
      const int r = x / kHdWords % kHdCols;
      const int t = x / (kHdWords * kHdCols);
      if (c0 + r < lenb && g0 + wd < groups)
        hdig[(t * lenb + c0 + r) * groups + g0 + wd] = sw[t][r][wd];
    }
    __syncthreads();
  }
  red[ky][cx] = zsum;
  __syncthreads();
  if (ky == 0 && ok) {
    for (int y = 1; y < kHdK; ++y) zsum += red[y][cx];
    hscale[c] = ldexp(1.0, -eh);
    hcorr[c] = kOffsetUnit * zsum;
    hdiag[c] = hcol[c * lenb + c];
  }
}

// GEMM tile: 128 M rows (64 alpha strings, real and imaginary rows) x 64
// columns per workgroup of 8 waves (4 x 2, 32 x 32 per wave: 2 x 2 MFMA
// tiles of 16 x 16, six accumulators each, 96 registers), two waves per
// SIMD, K in steps of 64.  With 64 x 32 per wave (192 accumulators, one
// wave per SIMD) the LDS operand reads per MFMA were fewer, but every wait
// for a K step's loads and fragments was exposed: 1.59 ms instead of 1.35
// at norb 14.
// The operand tiles are double-buffered in LDS (2 x 68 KB, one workgroup
// per CU) and filled by direct buffer-to-LDS loads (buffer_load_dwordx4
// ... lds: lane L of an instruction writes bytes 16 L .. 16 L + 15 past the
// instruction's LDS base), so no staging registers: one instruction moves
// 16 rows x 64 bytes of one digit plane.  Rows are 64 bytes (16 banks),
// unpadded; the four 16-byte chunks of row r sit XOR-swizzled by (r / 2) % 4,
// so each 8 lanes of a fragment read (rows r..r+7 at one chunk: even and odd
// rows on the two bank halves, the four rows of each parity on four chunks)
// cover the 32 banks once (keyed by (r / 4) % 4, rows r and r + 2 shared
// banks: 1.5-2% slower).
// Step ks + 1's loads go out after the barrier of step ks and land in the
// other buffer while step ks's MFMAs run; one wait and one barrier per
// step.
constexpr int kBdBuf = (6 * kBgTM + 5 * kBgTN) * kBgK;   // bytes per buffer
constexpr int kBdNoRow = 0x7ff00000;        // offset of a row past the matrix

__device__ __forceinline__ int bd_off(int row, int chunk) {
  return row * kBgK + 16 * (chunk ^ ((row >> 1) & 3));
}

typedef __attribute__((address_space(3))) void lds_void_t;

// TRANS: the left factor is C^T (lena, lenb exchanged by the caller), and the
// result is added to out at the transposed place.
template <bool TRANS>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
k_beta_gemm_oz(int64_t lena, int64_t lenb, int64_t ldk,
                  const uint8_t* __restrict__ cdig,
                  const double* __restrict__ cscale,
                  const uint8_t* __restrict__ hdig,
                  const double* __restrict__ hscale,
                  const double* __restrict__ hcorr,
                  const double* __restrict__ hdiag,
                  const double* __restrict__ coeff, double* __restrict__ out,
                  const int32_t* __restrict__ done, int tm, int tn,
                  int per_xcd) {
  // two buffers as two arrays: the compiler can tell the loads into one
  // from the fragment reads of the other
  __shared__ __align__(16) uint8_t buf0[kBdBuf];
  __shared__ __align__(16) uint8_t buf1[kBdBuf];
  if (done && *done) return;
  int im, in;
  if (!oz_tile(tm, tn, per_xcd, &im, &in)) return;
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int64_t rows = 2 * lena;
  const int64_t m0 = static_cast<int64_t>(im) * kBgTM;
  const int64_t n0 = static_cast<int64_t>(in) * kBgTN;
  const int wm = (wave >> 1) * 32;
  const int wn = (wave & 1) * 32;
  const __amdgpu_buffer_rsrc_t rcd = buffer_of(cdig, 6 * rows * ldk);
  const __amdgpu_buffer_rsrc_t rhd = buffer_of(hdig, 5 * lenb * ldk);
  // lane L of a load instruction: tile row r0 + L/4, LDS chunk L%4, which
  // holds global chunk (L%4) ^ ((L/8)%4) (r0 is a multiple of 16)
  const int lrow = lane >> 2;
  const int lq = (lane & 3) ^ ((lane >> 3) & 3);
  // C: 6 planes x 8 instructions of 16 rows; H: 5 planes x 4; wave w takes
  // instructions w, w + 8, ... (six C, and three or two H: waves 0..3 take
  // H instruction 16 + w)  Byte offsets at k0 = 0, once: a row past
  // the matrix gets kBdNoRow, which stays past the end of the digit planes
  // for every k0 (their size is below kBdNoRow), so it reads zero.
  int coff[6], hoff[3];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int ins = wave + 8 * j;
    const int i = ins >> 3, r0 = (ins & 7) * 16;
    const int64_t gr = m0 + r0 + lrow;
    coff[j] = gr < rows ? static_cast<int>((i * rows + gr) * ldk + 16 * lq) : kBdNoRow;
  }
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    const int ins = wave + 8 * j;
    const int i = ins >> 2, r0 = (ins & 3) * 16;
    const int64_t gn = n0 + r0 + lrow;
    hoff[j] = (ins < 20 && gn < lenb) ? static_cast<int>((i * lenb + gn) * ldk + 16 * lq) : kBdNoRow;
  }
  auto issue = [&](uint8_t* base, int k0) {
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      const int ins = wave + 8 * j;
      const int i = ins >> 3, r0 = (ins & 7) * 16;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rcd, (lds_void_t*)(base + (i * kBgTM + r0) * kBgK), 16, coff[j] + k0,
          0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int ins = wave + 8 * j;
      if (ins < 20) {
        const int i = ins >> 2, r0 = (ins & 3) * 16;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rhd, (lds_void_t*)(base + 6 * kBgTM * kBgK + (i * kBgTN + r0) * kBgK),
            16, hoff[j] + k0, 0, 0, 0);
      }
    }
  };
  int4v acc[2][2][6];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int m = 0; m < 6; ++m) acc[a][b][m] = int4v{0, 0, 0, 0};
  // both column tiles' Hbb fragments held, one row tile's C fragments at a
  // time (64 operand registers)
  auto compute = [&](const uint8_t* base) {
    const uint8_t* sc = base;
    const uint8_t* sh = base + 6 * kBgTM * kBgK;
    const int q = lane >> 4;
    int4v b[2][5];
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int i = 0; i < 5; ++i)
        b[y][i] = *reinterpret_cast<const int4v*>(
            sh + i * kBgTN * kBgK + bd_off(wn + 16 * y + (lane & 15), q));
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      int4v a[6];
#pragma unroll
      for (int i = 0; i < 6; ++i)
        a[i] = *reinterpret_cast<const int4v*>(
            sc + i * kBgTM * kBgK + bd_off(wm + 16 * x + (lane & 15), q));
#pragma unroll
      for (int y = 0; y < 2; ++y)
#pragma unroll
        for (int i = 0; i < 6; ++i)
#pragma unroll
          for (int t = 0; t < 5; ++t)
            if (t <= i)
              acc[x][y][i - t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                  a[i], b[y][t], acc[x][y][i - t], 0, 0, 0);
    }
  };
  const int nk = static_cast<int>(ldk / kBgK);
  issue(buf0, 0);
  for (int ks = 0; ks < nk; ++ks) {
    // step ks from one buffer; step ks + 1 loads into the other meanwhile
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    uint8_t* cur = (ks & 1) ? buf1 : buf0;
    uint8_t* nxt = (ks & 1) ? buf0 : buf1;
    if (ks + 1 < nk) issue(nxt, (ks + 1) * kBgK);
    compute(cur);
  }
  // output item e of lane l: M row 4 (l/16) + e, column l%16; rows 2 Ia
  // (real) and 2 Ia + 1 (imaginary) are items e and e + 1
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int64_t col = n0 + wn + 16 * y + (lane & 15);
      if (col >= lenb) continue;
      const double hs = hscale[col];
      const double hc = hcorr[col];
      const double hd = hdiag[col];
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        const int64_t row = m0 + wm + 16 * x + 4 * (lane >> 4) + e;
        if (row >= rows) continue;
        const int64_t ia = row >> 1;
        double v[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          double t = static_cast<double>(acc[x][y][5][e + c]);
#pragma unroll
          for (int m = 4; m >= 0; --m)
            t = fma(t, 256.0, static_cast<double>(acc[x][y][m][e + c]));
          v[c] = fma(t, 4294967296.0, hc) * hs;
        }
        const double cs = cscale[ia];
        const int64_t at = TRANS ? col * lena + ia : ia * lenb + col;
        const double2 x0 = reinterpret_cast<const double2*>(coeff)[at];
        double2* dst = reinterpret_cast<double2*>(out) + at;
        double2 o = TRANS ? *dst : make_double2(0.0, 0.0);
        o.x += fma(v[0], cs, hd * x0.x);
        o.y += fma(v[1], cs, hd * x0.y);
        *dst = o;
      }
    }
}

}  // namespace

int64_t beta_oz_ldk(int64_t lenb) { return (lenb + kBgK - 1) / kBgK * kBgK; }

// C digit planes of the apply: 6 x 2 lena x ldk bytes, then lena doubles.
int64_t beta_oz_workspace_bytes(int64_t lena, int64_t lenb) {
  return 6 * 2 * lena * beta_oz_ldk(lenb) + 8 * lena;
}

bool beta_oz_shape_ok(int64_t lena, int64_t lenb) {
  // byte offsets into the digit planes stay below the out-of-range row
  // offset of k_beta_gemm_oz
  const int64_t lim = kBdNoRow - beta_oz_ldk(lenb);
  return lenb < 26214 && 6 * 2 * lena * beta_oz_ldk(lenb) < lim &&
         5 * lenb * beta_oz_ldk(lenb) < lim;
}

namespace {

// The GEMM of the digits of len_m data rows with those of H (len_n x len_n).
template <bool TRANS>
void digit_gemm(int64_t len_m, int64_t len_n, const uint8_t* cdig,
                const double* cscale, const void* hoz, const double* coeff,
                double* out, hipStream_t st, const int32_t* done) {
  const int64_t ldk = beta_oz_ldk(len_n);
  const uint8_t* hdig = static_cast<const uint8_t*>(hoz);
  const double* hscale = reinterpret_cast<const double*>(hdig + 5 * len_n * ldk);
  const int tm = static_cast<int>((2 * len_m + kBgTM - 1) / kBgTM);
  const int tn = static_cast<int>((len_n + kBgTN - 1) / kBgTN);
  const int per_xcd = (tm * tn + kBgXcds - 1) / kBgXcds;
  k_beta_gemm_oz<TRANS><<<static_cast<unsigned>(per_xcd * kBgXcds), 512, 0, st>>>(
      len_m, len_n, ldk, cdig, cscale, hdig, hscale, hscale + len_n,
      hscale + 2 * len_n, coeff, out, done, tm, tn, per_xcd);
}

}  // namespace

int launch_beta_gemm_oz(int64_t lena, int64_t lenb, const void* hoz,
                        const double* coeff, const double* rowmax,
                        void* cwork, double* out, hipStream_t st,
                        const int32_t* done) {
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  const int64_t ldk = beta_oz_ldk(lenb);
  uint8_t* cdig = static_cast<uint8_t*>(cwork);
  double* cscale = reinterpret_cast<double*>(cdig + 6 * 2 * lena * ldk);
  const int64_t nthr = lena * (ldk / 4);
  k_c_digits<<<blocks_for(nthr, 256), 256, 0, st>>>(
      lena, lenb, ldk, coeff, rowmax, reinterpret_cast<uint32_t*>(cdig), cscale,
      done);
  FQEHIP_CHECK_LAUNCH("k_c_digits");
  digit_gemm<false>(lena, lenb, cdig, cscale, hoz, coeff, out, st, done);
  FQEHIP_CHECK_LAUNCH("k_beta_gemm_oz");
  return FQEHIP_OK;
}

// out += Haa C, on the digits of C^T (in cwork, beta_oz_workspace_bytes(lenb,
// lena) bytes); colmax: the column maxima of |C|.
int launch_alpha_gemm_oz(int64_t lena, int64_t lenb, const void* hoz,
                         const double* coeff, const double* colmax, void* cwork,
                         double* out, hipStream_t st, const int32_t* done) {
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  const int64_t ldk = beta_oz_ldk(lena);
  uint8_t* cdig = static_cast<uint8_t*>(cwork);
  double* cscale = reinterpret_cast<double*>(cdig + 6 * 2 * lenb * ldk);
  // every word of the ldk bytes of a row is written: the grid covers ldk / 64
  const dim3 grid(blocks_for(lenb, kCtB), static_cast<unsigned>(ldk / kCtA));
  k_ct_digits<<<grid, 256, 0, st>>>(lena, lenb, ldk, coeff, colmax,
                                    reinterpret_cast<uint32_t*>(cdig), cscale, done);
  FQEHIP_CHECK_LAUNCH("k_ct_digits");
  digit_gemm<true>(lenb, lena, cdig, cscale, hoz, coeff, out, st, done);
  FQEHIP_CHECK_LAUNCH("k_beta_gemm_oz");
  return FQEHIP_OK;
}

// Row maxima of |C|, with colmax its column maxima; zeroes nsum sums.
int launch_absmax(int64_t lena, int64_t lenb, const double* coeff,
                  double* rowmax, double* colmax, double* sums, int64_t nsum,
                  hipStream_t st, const int32_t* done) {
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  const unsigned grid = static_cast<unsigned>(lena < 65536 ? lena : 65536);
  unsigned long long* cm = reinterpret_cast<unsigned long long*>(colmax);
  k_row_absmax<<<grid, 256, 0, st>>>(lena, lenb, coeff, rowmax, cm,
                                     reinterpret_cast<unsigned long long*>(sums), nsum, done);
  FQEHIP_CHECK_LAUNCH("k_row_absmax");
  if (!colmax) return FQEHIP_OK;
  const dim3 cgrid(blocks_for(lenb, 256), blocks_for(lena, kColRows));
  k_col_absmax<<<cgrid, 256, 0, st>>>(lena, lenb, coeff, cm, done);
  FQEHIP_CHECK_LAUNCH("k_col_absmax");
  return FQEHIP_OK;
}

}  // namespace fqehip

using namespace fqehip;

extern "C" int64_t fqehip_beta_block_digits_bytes(int64_t lenb) {
  if (lenb < 0) return -1;
  return 5 * lenb * beta_oz_ldk(lenb) + 24 * lenb;
}

extern "C" int fqehip_beta_block_digits(int64_t lenb, const double* d_hcol,
                                        void* d_hoz, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(lenb >= 0, "lenb=%lld", static_cast<long long>(lenb));
  if (lenb == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_hcol && d_hoz, "NULL pointer");
  FQEHIP_CHECK_ARG(beta_oz_shape_ok(1, lenb), "lenb=%lld too large",
                   static_cast<long long>(lenb));
  hipStream_t st = as_stream(stream);
  const int64_t ldk = beta_oz_ldk(lenb);
  uint32_t* hdig = static_cast<uint32_t*>(d_hoz);
  double* hscale = reinterpret_cast<double*>(static_cast<uint8_t*>(d_hoz) + 5 * lenb * ldk);
  double* hcorr = hscale + lenb;
  k_hbb_digits<<<blocks_for(lenb, kHdCols), kHdCols * kHdK, 0, st>>>(
      lenb, ldk, d_hcol, hdig, hscale, hcorr, hcorr + lenb);
  FQEHIP_CHECK_LAUNCH("k_hbb_digits");
  return FQEHIP_OK;
}

extern "C" int fqehip_beta_gemm_digits(int64_t lena, int64_t lenb,
                                       const void* d_hoz, const void* d_coeff,
                                       void* d_work, void* d_out,
                                       const int32_t* d_done, void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(lena >= 0 && lenb >= 0, "negative size");
  if (lena == 0 || lenb == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_hoz && d_coeff && d_work && d_out, "NULL pointer");
  FQEHIP_CHECK_ARG(beta_oz_shape_ok(lena, lenb), "sector too large");
  hipStream_t st = as_stream(stream);
  double* rowmax = static_cast<double*>(d_work);
  int rc = launch_absmax(lena, lenb, static_cast<const double*>(d_coeff),
                         rowmax, nullptr, nullptr, 0, st, d_done);
  if (rc) return rc;
  return launch_beta_gemm_oz(lena, lenb, d_hoz,
                             static_cast<const double*>(d_coeff), rowmax,
                             rowmax + lena, static_cast<double*>(d_out), st,
                             d_done);
}

extern "C" int64_t fqehip_pull_digits_bytes(int npull) {
  if (npull < 0) return -1;
  return npull * (kWDigBytes + static_cast<int64_t>(kOzQ) * 8) + sizeof(OzUnit);
}

extern "C" int fqehip_pull_digits(int npull, const double* d_w, void* d_woz,
                                  void* stream) {
  clear_error();
  FQEHIP_CHECK_ARG(npull >= 0 && npull <= kOzQ, "npull=%d outside 0..%d", npull, kOzQ);
  if (npull == 0) return FQEHIP_OK;
  FQEHIP_CHECK_ARG(d_w && d_woz, "NULL pointer");
  uint8_t* dig = static_cast<uint8_t*>(d_woz);
  double* z = reinterpret_cast<double*>(dig + npull * kWDigBytes);
  OzUnit* unit = reinterpret_cast<OzUnit*>(z + static_cast<int64_t>(npull) * kOzQ);
  k_pull_digits<<<npull, kOzQ, 0, as_stream(stream)>>>(npull, d_w, dig, z, unit);
  FQEHIP_CHECK_LAUNCH("k_pull_digits");
  return FQEHIP_OK;
}
