// Partial rows summed in a fixed order and scattered to the caller's order.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sgpp_hip {

namespace {

// The sum of rows [0, nrows) of p[row * ld], by the kRows * kCols threads of a
// block: kRows threads take a column's rows in turn, eight loads in flight each,
// and their sums are added in a fixed order. Complete in threads [0, kCols).
constexpr int kRows = 8;
constexpr int kCols = 64;
__device__ __forceinline__ double sum_rows(const double* __restrict__ p, int64_t ld, int nrows) {
  __shared__ double s[kRows][kCols];
  const int c = threadIdx.x % kCols, q = threadIdx.x / kCols;
  double sum = 0.0;
  int r = q;
  for (; r + 7 * kRows < nrows; r += 8 * kRows) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[static_cast<int64_t>(r + u * kRows) * ld];
#pragma unroll
    for (int u = 0; u < 8; ++u) sum += v[u];
  }
  for (; r < nrows; r += kRows) sum += p[static_cast<int64_t>(r) * ld];
  s[q][c] = sum;
  __syncthreads();
  if (q == 0)
#pragma unroll
    for (int u = 1; u < kRows; ++u) sum += s[u][c];
  return sum;
}

// out[to[i]] = the sum of rows [0, nrows) of part[.][i], for to[i] >= 0
__global__ __launch_bounds__(kRows* kCols) void reduce_rows_kernel(
    const double* __restrict__ part, int64_t ld, int nrows, const int32_t* __restrict__ to,
    double* __restrict__ out, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kCols + threadIdx.x % kCols;
  const double sum = sum_rows(part + (i < n ? i : 0), ld, i < n ? nrows : 0);
  if (threadIdx.x >= kCols || i >= n) return;
  const int32_t j = to[i];
  if (j >= 0) out[j] = sum;
}

inline unsigned blocks(int64_t n, int b) { return static_cast<unsigned>((n + b - 1) / b); }

}  // namespace

}  // namespace sgpp_hip
