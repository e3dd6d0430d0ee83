// sdm_reduce.h -- sums of per-block partial records in float64 and in a fixed order, shared by the backward kernels.
#pragma once
#include "sdm_common.h"

namespace sdmrt {

// The sum over n_rec records of part[r * rec_stride + i] for item i (nothing where !live), in float64: block of 64 x 16
// threads, lane l of group rg sums records rg, rg + 16, ... of its item (loads issued together), then the 16 group
// sums are added in group order: a fixed order, so the result is deterministic.  Every thread calls it; the sums are
// returned in group 0's lanes.  red: 16 x 64 doubles of LDS, free again after the next __syncthreads
constexpr int kRedGroups = 16;

template <typename T>
__device__ __forceinline__ double reduce_item(const T* __restrict__ part, int n_rec, int64_t rec_stride, int64_t i,
                                              bool live, double (*red)[64]) {
  const int l = threadIdx.x & 63;
  const int rg = threadIdx.x >> 6;
  double s = 0.0;
  if (live) {
    constexpr int kBatch = 16;
    for (int r0 = rg; r0 < n_rec; r0 += kRedGroups * kBatch) {
      T v[kBatch];
#pragma unroll
      for (int q = 0; q < kBatch; ++q) {
        const int r = r0 + q * kRedGroups;
        v[q] = r < n_rec ? part[static_cast<int64_t>(r) * rec_stride + i] : T(0);
      }
#pragma unroll
      for (int q = 0; q < kBatch; ++q) s += static_cast<double>(v[q]);
    }
  }
  red[rg][l] = s;
  __syncthreads();
  double t = 0.0;
  if (rg == 0)
    for (int q = 0; q < kRedGroups; ++q) t += red[q][l];
  return t;
}

// out[i] = the sum over records of item i, for n_items items
template <typename T>
__global__ void __launch_bounds__(64 * kRedGroups) reduce_records_kernel(const T* __restrict__ part, int n_rec,
                                                                        int64_t rec_stride, int64_t n_items,
                                                                        float* __restrict__ out) {
  __shared__ double red[kRedGroups][64];
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + (threadIdx.x & 63);
  const double t = reduce_item(part, n_rec, rec_stride, i, i < n_items, red);
  if (threadIdx.x < 64 && i < n_items) out[i] = static_cast<float>(t);
}

}  // namespace sdmrt
