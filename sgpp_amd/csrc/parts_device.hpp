// Small kernels around the tree and hit-list products: right-hand sides into
// storage order, partial rows summed and scattered to the caller's order.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sgpp_hip {

namespace {

// Y[m] = y[dperm[m]] for stored row m, 0 for the padding rows
template <typename T>
__global__ void prep_rows_kernel(const double* __restrict__ y, const int32_t* __restrict__ dperm,
                                   T* __restrict__ Y, int64_t n, int64_t npad) {
  const int64_t m = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (m < npad) Y[m] = m < n ? static_cast<T>(y[dperm[m]]) : T(0);
}

// out[to[i]] = (scale ? scale[i] : 1) times the sum of rows [0, nrows) of
// part[.][i], for to[i] >= 0.
// kRows threads take a column's rows in turn, eight loads in flight each, and
// their sums are added in a fixed order.
constexpr int kRows = 8;
constexpr int kCols = 64;
__global__ __launch_bounds__(kRows* kCols) void reduce_rows_kernel(
    const double* __restrict__ part, int64_t ld, int nrows, const int32_t* __restrict__ to,
    const double* __restrict__ scale, double* __restrict__ out, int64_t n) {
  __shared__ double s[kRows][kCols];
  const int c = threadIdx.x % kCols, q = threadIdx.x / kCols;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * kCols + c;
  double sum = 0.0;
  if (i < n) {
    const double* p = part + i;
    int r = q;
    for (; r + 7 * kRows < nrows; r += 8 * kRows) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = p[static_cast<int64_t>(r + u * kRows) * ld];
#pragma unroll
      for (int u = 0; u < 8; ++u) sum += v[u];
    }
    for (; r < nrows; r += kRows) sum += p[static_cast<int64_t>(r) * ld];
  }
  s[q][c] = sum;
  __syncthreads();
  if (q == 0 && i < n) {
#pragma unroll
    for (int u = 1; u < kRows; ++u) sum += s[u][c];
    const int32_t j = to[i];
    if (j >= 0) out[j] = scale ? sum * scale[i] : sum;
  }
}

inline unsigned blocks(int64_t n, int b) { return static_cast<unsigned>((n + b - 1) / b); }

}  // namespace

}  // namespace sgpp_hip
