// Shared by the pull-form kernels (pull.hip, ozaki.hip) and their callers
// (apply.hip, batch.hip).
#pragma once

#include "fqehip_common.h"

namespace fqehip {

// The convergence test of a Taylor series' last term, made by the next term's
// row kernel (partials NULL: none).
constexpr int64_t kSeriesRows = 1024;      // partials a wave reads at most
struct PullSeries {
  const double* partials = nullptr;        // |row|^2 of the last term
  double accuracy = 0.0;
  int term = 0;                            // its number
  double* norm = nullptr;
  int32_t* nterms = nullptr;
  int32_t* done = nullptr;
};

// What a row kernel does with the finished row of H C: nothing (out NULL: the
// row accumulators keep it), or out = alpha (H C) + beta cin, acc += out,
// partials[ia] = |out row|^2.
struct PullEpilogue {
  double alpha_re = 1.0, alpha_im = 0.0, beta_re = 0.0, beta_im = 0.0;
  const double* cin = nullptr;
  double* out = nullptr;
  double* acc = nullptr;
  double* partials = nullptr;
  PullSeries series;
};

// Launch shape of a batch group of pull-form sectors (one class).
struct PullGroupLaunch {
  int cls, nsec, rows, tiles;
  size_t lds;
  bool any_apply;
};

bool pull_supported(const fqehip_sector* s);
// Whether an FP64 apply of the sector is the row kernel alone (which then also
// takes the test of a series).
bool pull_one_launch(const fqehip_sector* s);
int launch_same_spin(const fqehip_sector* s, int complex_op,
                     const double* coeff, double* rowacc,
                     const PullSeries& series, hipStream_t st,
                     const int32_t* done);
int launch_pull_rows(const fqehip_sector* s, int complex_op,
                     const double* coeff, double* rowacc,
                     const PullEpilogue& e, hipStream_t st, const int32_t* done);
int pull_group_class(const fqehip_sector* s);
size_t pull_group_bytes(int nsec);
int pull_group_fill(const fqehip_batch_item* const* items, const int64_t* spare,
                    int nsec, void* host, PullGroupLaunch* g);
int launch_pull_group(const PullGroupLaunch& g, const void* d_secs, int step,
                      double ar, double ai, hipStream_t st);

bool pull_oz_supported(const fqehip_sector* s);
int pull_oz_segments(const fqehip_sector* s);
int launch_pull_rows_oz(const fqehip_sector* s, const double* coeff,
                        const double* rowmax, double* rowacc, double* sums,
                        const PullEpilogue& e, hipStream_t st,
                        const int32_t* done);

// Defined in apply.hip: whether the sector's two-body applies run in the pull
// form, whether with digit rows, and where its workspace holds a second term
// buffer (byte offset; 16 lena lenb bytes).
bool pull_sector(int precision, const fqehip_sector* s);
bool digit_rows(const fqehip_sector* s);
int64_t pull_spare_offset(const fqehip_sector* s);

// partial[0] = the workgroup's sum of v, in a fixed order; smem holds a double
// per wave and is free.
__device__ __forceinline__ void row_norm(double v, double* partial, char* smem) {
  double* red = reinterpret_cast<double*>(smem);
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (unsigned w = 0; w < blockDim.x / 64; ++w) t += red[w];
    *partial = t;
  }
}

// The test after a term of a Taylor series, by every wave for itself at the
// start of the next term's first kernel (a kernel of its own costs as much as
// the rows of a small sector): the norm of the last term from its row partials,
// stored with the term count by the first workgroup.  A wave that already
// finds the flag set by that workgroup returns as the test would tell it.
__device__ __forceinline__ bool series_done(const PullSeries& q, int lena) {
  const int lane = threadIdx.x & 63;
  double s = 0.0;
  for (int k = lane; k < lena; k += 64) s += q.partials[k];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) s += __shfl_xor(s, o);
  const double nrm = sqrt(s);
  const bool done = nrm < q.accuracy;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *q.norm = nrm;
    *q.nterms = q.term;
    if (done) *q.done = 1;
  }
  return done;
}

}  // namespace fqehip
