// sdm_reduce.h -- sums of per-block partial records in float64 and in a fixed order, shared by the backward kernels.
#pragma once
#include "sdm_common.h"

namespace sdmrt {

// Sums over records: out[i] = sum_r part[r * rec_stride + i] (r < n_rec) in float64 for n_items items.  Block of
// 64 x 16 threads: lane i of group rg sums records rg, rg + 16, ... (loads issued together), then the 16 group sums
// are added in group order: a fixed order, so the result is deterministic.
constexpr int kRedGroups = 16;

template <typename T, typename OutT = double>
__global__ void __launch_bounds__(64 * kRedGroups) reduce_records_kernel(const T* __restrict__ part, int n_rec,
                                                                        int64_t rec_stride, int64_t n_items,
                                                                        OutT* __restrict__ out) {
  __shared__ double red[kRedGroups][64];
  const int l = threadIdx.x & 63;
  const int rg = threadIdx.x >> 6;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 64 + l;
  double s = 0.0;
  if (i < n_items) {
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
  if (rg == 0 && i < n_items) {
    double t = 0.0;
    for (int q = 0; q < kRedGroups; ++q) t += red[q][l];
    out[i] = static_cast<OutT>(t);
  }
}

}  // namespace sdmrt
