// Kernels of the subspace tree (tree_device.hpp). Included by one source file
// per compute type and basis, so that they compile in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include "cull_device.hpp"
#include "tree_device.hpp"

#pragma clang diagnostic ignored "-Wint-to-pointer-cast"

namespace sgpp_hip {

namespace {

// a record as one vector: off, ctl, scale, pad (scalar loads)
typedef unsigned TreeRecWords __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(4))) TreeRecWords* TreeRecPtr;

// one instruction each: the C++ forms add a range check or a canonicalisation
__device__ __forceinline__ unsigned to_fixed(float x) {  // floor(x 2^32), 2^32 - 1 at x = 1
  unsigned r;
  const float s = x * 4294967296.0f;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(s));
  return r;
}
__device__ __forceinline__ unsigned to_fixed(double x) {
  unsigned r;
  const double s = x * 4294967296.0;
  asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(s));
  return r;
}
__device__ __forceinline__ float max_raw(float a, float b) {
  float r;
  asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_raw(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float min_raw(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double min_raw(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float rint_raw(float a) { return __builtin_rintf(a); }
__device__ __forceinline__ double rint_raw(double a) { return __builtin_rint(a); }
__device__ __forceinline__ float scale_of(uint32_t bits, float) { return __uint_as_float(bits); }
__device__ __forceinline__ double scale_of(uint32_t bits, double) {
  return __hiloint2double(static_cast<int>(bits), 0);
}

// the level-1 hat at x
template <typename T>
__device__ __forceinline__ T level_one(T x) {
  return min_raw(x + x, T(2) - (x + x));
}

// Values indexed by a wave-uniform dimension, in registers: 32-bit words in
// vectors (an indexed register move per word; of fewer than nine elements the
// compiler would select by a chain of compares, twice the walk's other work at
// eight dimensions). More than 16 dimensions are two vectors, the even and the
// odd ones (split at the middle, the index into the upper half became a lane
// value, and each read a loop over its lanes: 36 scalar instructions a record).
template <typename T, int DB>
struct DimRegs {
  static constexpr int kWords = sizeof(T) / 4;
  static constexpr bool kTwo = DB > 16;
  static constexpr int kSize = DB <= 9 ? 9 : (kTwo ? DB / 2 : DB);
  typedef unsigned Vec __attribute__((ext_vector_type(kSize)));
  Vec a[kTwo ? 2 : 1][kWords];
  __device__ __forceinline__ void set(int d, T v) {  // d known at compile time
    unsigned w[kWords];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < kWords; ++i) a[kTwo ? d & 1 : 0][i][kTwo ? d >> 1 : d] = w[i];
  }
  __device__ __forceinline__ T get(int part, int i) const {  // part known at compile time
    unsigned w[kWords];
#pragma unroll
    for (int j = 0; j < kWords; ++j) w[j] = a[part][j][i];
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
  }
};
// out[.][k] = v[.][k] of dimension r
template <typename T, int DB, int K, int N>
__device__ __forceinline__ void dim_values(const DimRegs<T, DB> (*const (&v)[N])[K], int r,
                                           T (*const (&out)[N])[K]) {
  auto read = [&](int part, int i) {
    __builtin_amdgcn_sched_barrier(0);  // (one indexed-register mode for all the moves)
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int k = 0; k < K; ++k) (*out[n])[k] = (*v[n])[k].get(part, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (!DimRegs<T, DB>::kTwo)
    read(0, r);
  else if (r & 1)
    read(1, r >> 1);
  else
    read(0, r >> 1);
}
template <typename T, int DB, int K>
__device__ __forceinline__ void dim_values(const DimRegs<T, DB> (&v)[K], int r, T (&out)[K]) {
  const DimRegs<T, DB>(*const vs[1])[K] = {&v};
  T(*const outs[1])[K] = {&out};
  dim_values<T, DB, K, 1>(vs, r, outs);
}

// The data points of a walk: coordinates in registers (DB > 0), and for
// Linear grids the products rest[d] of the level-1 factors of the dimensions
// after d; or (DB == 0, many dimensions) read from memory when a run begins.
// one[k]: the product of all level-1 factors (1 for ModLinear).
template <typename T, int DB, int K, bool kMod>
struct TreePoints {
  DimRegs<T, DB> x[K];
  DimRegs<T, DB> rest[kMod ? 1 : K];
  __device__ __forceinline__ void load(const T* __restrict__ X, int64_t ldx, int D, int64_t m,
                                       T (&one)[K]) {
    T v[K][DB];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int k = 0; k < K; ++k) v[k][d] = d < D ? X[d * ldx + m + k * 64] : T(0.5);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      one[k] = T(1);
#pragma unroll
      for (int d = DB - 1; d >= 0; --d) {
        x[k].set(d, v[k][d]);
        if constexpr (!kMod) {
          rest[k].set(d, one[k]);
          one[k] *= level_one(v[k][d]);  // (1 at the unused dimensions' 1/2)
        }
      }
    }
  }
  __device__ __forceinline__ void coordinates(int r, T (&xr)[K]) const {
    dim_values(x, r, xr);
  }
  // the level-1 factors after dimension r
  __device__ __forceinline__ void after(int r, int, T (&s)[K]) const { dim_values(rest, r, s); }
};
template <typename T, int K, bool kMod>
struct TreePoints<T, 0, K, kMod> {
  const T* p;
  int64_t ld;
  __device__ __forceinline__ void load(const T* __restrict__ X, int64_t ldx, int D, int64_t m,
                                       T (&one)[K]) {
    p = X + m;
    ld = ldx;
#pragma unroll
    for (int k = 0; k < K; ++k) one[k] = T(1);
    if constexpr (!kMod) after(-1, D, one);
  }
  __device__ __forceinline__ void coordinates(int r, T (&xr)[K]) const {
#pragma unroll
    for (int k = 0; k < K; ++k) xr[k] = p[r * ld + k * 64];
  }
  __device__ __forceinline__ void after(int r, int D, T (&s)[K]) const {
#pragma unroll
    for (int k = 0; k < K; ++k) s[k] = T(1);
    for (int d = D - 1; d > r; --d)
#pragma unroll
      for (int k = 0; k < K; ++k) s[k] *= level_one(p[d * ld + k * 64]);
  }
};

// The walk over a chunk's program. Per depth the parent's product R (of the
// factors of the dimensions up to its last step; for Linear grids extended by
// the level-1 factors of the dimensions passed since) and table position F. A
// run (the children of one parent in one dimension) fetches x, its 32-bit
// fixed-point form (the cell of level l is its top l - 1 bits) and rr, the
// product of all factors but the run's own. Per node and data point:
//   t = 2^(l-1) x - 1/2, w = t - rint(t) in [-1/2, 1/2]: the hat is 1 - 2|w|
//   ModLinear: its extrapolated boundary functions are 2 - 2^l min(x, 1-x),
//   which exceeds the hat in the boundary cells only: the larger of the two.
// A point on a cell edge may round to either side: the hat is 0 there.
template <typename T, int DB, int K, bool kMod, int MD, typename Use>
struct TreeWalk {
  TreePoints<T, DB, K, kMod>& pts;
  Use& use;
  TreeRecPtr next;
  TreeRecWords cur;
  int D;
  T xr[K], rr[K], xm[K];
  unsigned fx[K];

  __device__ __forceinline__ void run(TreeRecPtr recs, const T (&R0)[K]) {
    next = recs;
    cur = next[0];
    unsigned F0[K];
#pragma unroll
    for (int k = 0; k < K; ++k) F0[k] = 0u;
    level<0>(R0, F0);
  }

  template <int kDepth>
  __device__ __forceinline__ void level(const T (&R0)[K], const unsigned (&F)[K]) {
    T R[K];
#pragma unroll
    for (int k = 0; k < K; ++k) R[k] = R0[k];
    for (;;) {
      const unsigned off = cur.x, ctl = cur.y, scale = cur.z, from = cur.w;
      ++next;
      cur = next[0];  // in flight during this node
      if (ctl & kTreeRun) {
        const int r = (ctl >> kTreeDimShift) & 63u;
        if constexpr (!kMod) {
          for (int d = static_cast<int>(from); d < r; ++d) {
            pts.coordinates(d, xr);
#pragma unroll
            for (int k = 0; k < K; ++k) R[k] *= level_one(xr[k]);
          }
          pts.after(r, D, rr);
        }
        pts.coordinates(r, xr);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          fx[k] = to_fixed(xr[k]);
          rr[k] = kMod ? R[k] : R[k] * rr[k];
          if constexpr (kMod) xm[k] = level_one(xr[k]);
        }
      }
      unsigned E[K];
#pragma unroll
      for (int k = 0; k < K; ++k) E[k] = __builtin_amdgcn_alignbit(F[k], fx[k], ctl);
      use.begin(off, ctl, E);
      const T L = scale_of(scale, T(0));
      T f[K], P[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const T t = fmaT(xr[k], L, T(-0.5));
        const T w = t - rint_raw(t);
        f[k] = fmaT(T(-2), absT(w), T(1));
        if constexpr (kMod) f[k] = max_raw(f[k], fmaT(-L, xm[k], T(2)));
        P[k] = rr[k] * f[k];
      }
      use.end(off, ctl, P, E);
      if (ctl & (kTreePush | kTreeLast | kTreeFlush)) {
        if (sizeof(T) == 4 && (ctl & kTreeFlush)) use.flush();
        if constexpr (kDepth + 1 < MD)
          if (ctl & kTreePush) {
            if constexpr (!kMod)
#pragma unroll
              for (int k = 0; k < K; ++k) P[k] = R[k] * f[k];
            level<kDepth + 1>(P, E);
          }
        if (ctl & kTreeLast) return;
      }
    }
  }
};

extern __shared__ __align__(16) unsigned char tree_lds[];

// byte address in LDS (the kernels have no LDS but tree_lds, which begins at 0)
template <typename T>
__device__ __forceinline__ T lds_read(unsigned a) {
  typedef const __attribute__((address_space(3))) T* Ptr;
  return *(Ptr)(a);
}

// mult: the node's weight at the point's table position, from the chunk's
// tables in LDS; read when the position is known, used after the products.
template <typename T, int K>
struct TreeGather {
  T acc[K], w[K];
  double accd[K];
  unsigned part0, partn, zero_off;
  __device__ __forceinline__ void begin(uint32_t off, uint32_t ctl, const unsigned (&E)[K]) {
    unsigned a[K];
#pragma unroll
    for (int k = 0; k < K; ++k) a[k] = E[k] * static_cast<unsigned>(sizeof(T)) + off;
    if (!(ctl & kTreeTable)) {
      // no table, or positions [part0, part0 + partn) of one
#pragma unroll
      for (int k = 0; k < K; ++k)
        a[k] = (ctl & kTreePart) && E[k] - part0 < partn ? a[k] : zero_off;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) w[k] = lds_read<T>(a[k]);
  }
  __device__ __forceinline__ void end(uint32_t, uint32_t, const T (&P)[K], const unsigned (&)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = fmaT(w[k], P[k], acc[k]);
  }
  __device__ __forceinline__ void flush() {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      accd[k] += static_cast<double>(acc[k]);
      acc[k] = T(0);
    }
  }
};

// mult: bound by vector instructions, ten to fourteen per node and data point
// (one scalar instruction issues in four cycles, so several points per lane
// share a node's); the weights of a chunk's subspaces are gathered from LDS,
// where up to 64 cells meet no bank conflict. Against evaluating every
// dimension of each grid point that a wave's box meets (kernel times): FP32,
// Linear d=8 level 6, 5e5 data points 1,028 to 260 us; FP64, the same 1,452 to
// 440 us, ModLinear d=7 level 6, 2.5e5 points 360 to 147 us, Linear d=30 level
// 3, 5e4 points 1,262 to 131 us.
template <typename T, int DB, int K, bool kMod, int MD>
__global__ __launch_bounds__(kTreeBlock) __attribute__((amdgpu_waves_per_eu(kMod ? 4 : 3)))
void tree_mult_kernel(const TreeMultArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t m = static_cast<int64_t>(blockIdx.x) * blockDim.x * K + wave * 64 * K + lane;
  T* lds = reinterpret_cast<T*>(tree_lds);
  TreePoints<T, DB, K, kMod> pts;
  T all[K], one[K];
  pts.load(static_cast<const T*>(a.X), a.ldx, a.D, m, all);
  TreeGather<T, K> g;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    g.acc[k] = T(0);
    g.accd[k] = 0.0;
    one[k] = T(1);
  }
  g.zero_off = a.zero_off;
  const int g0 = blockIdx.y * a.gper;
  const int c1 = a.groups[min(g0 + a.gper, a.ngroups)];
  for (int c = a.groups[g0]; c < c1; ++c) {
    const TreeChunk ch = a.chunks[c];
    __syncthreads();  // every wave is done with the last chunk's tables
    if (a.W) {
      const T* w = static_cast<const T*>(a.W) + ch.off0;
      for (int i = threadIdx.x; i < ch.n; i += blockDim.x) lds[i] = w[i];
    } else {
      const int32_t* ti = a.ti + ch.off0;
      for (int i = threadIdx.x; i < ch.n; i += blockDim.x) {
        const int32_t j = ti[i];
        lds[i] = j >= 0 ? static_cast<T>(a.alpha[j]) : T(0);
      }
    }
    if (threadIdx.x == 0) *reinterpret_cast<T*>(tree_lds + a.zero_off) = T(0);
    __syncthreads();
    g.part0 = ch.part0;
    g.partn = ch.n;
    if (ch.root) {
      const T w = lds[0];
#pragma unroll
      for (int k = 0; k < K; ++k) g.accd[k] += static_cast<double>(kMod ? w : w * all[k]);
    }
    if (ch.nrec > 0) {
      TreeWalk<T, DB, K, kMod, MD, TreeGather<T, K>> walk{pts, g, nullptr, TreeRecWords{}, a.D};
      walk.run((TreeRecPtr)(a.recs + ch.rec0), one);
      g.flush();
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double r = g.accd[k];
    const int64_t row = m + k * 64;
    if (a.part)
      a.part[static_cast<int64_t>(blockIdx.y) * a.ldx + row] = r;
    else if (row < a.M)
      a.out[a.dperm[row]] = r;
  }
}

// multTranspose: the sums over the wave's data points of each table position
// they fall in. Morton order puts most waves into one or two positions of a
// subspace: per position, the lanes' points are added, summed over the lanes
// (DPP) and added to the wave's own tables in LDS, in FP64 and in a fixed
// order (repeats are bit-identical).
template <typename T, int K>
struct TreeScatter {
  unsigned part0, partn;
  int lane;
  __device__ __forceinline__ void begin(uint32_t, uint32_t, const unsigned (&)[K]) {}
  __device__ __forceinline__ void flush() {}
  __device__ __forceinline__ void add(unsigned byte, T c) {
    const T s = sum_to_lane63(c);
    if (lane == 63)
      atomicAdd(reinterpret_cast<double*>(tree_lds + byte), static_cast<double>(s));
  }
  __device__ __forceinline__ void end(uint32_t off, uint32_t ctl, const T (&P)[K],
                                      const unsigned (&E)[K]) {
    unsigned long long rem[K];
    if (!(ctl & kTreeTable)) {
      if (!(ctl & kTreePart)) return;
#pragma unroll
      for (int k = 0; k < K; ++k) rem[k] = __ballot(E[k] - part0 < partn);
    } else {
      const unsigned e0 =
          static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(E[0])));
      unsigned long long other = 0ull;
#pragma unroll
      for (int k = 0; k < K; ++k) {
        rem[k] = ~0ull;
        other |= __ballot(E[k] != e0);
      }
      if (other == 0ull) {
        T c = P[0];
#pragma unroll
        for (int k = 1; k < K; ++k) c += P[k];
        add(off + e0 * 8u, c);
        return;
      }
    }
    for (;;) {
      unsigned e0 = 0u;
      bool any = false;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (!any && rem[k] != 0ull) {
          any = true;
          e0 = static_cast<unsigned>(__builtin_amdgcn_readlane(
              static_cast<int>(E[k]), __builtin_ctzll(rem[k])));
        }
      if (!any) break;
      T c = T(0);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const bool in = E[k] == e0;
        rem[k] &= ~__ballot(in);
        c += in ? P[k] : T(0);
      }
      add(off + e0 * 8u, c);
    }
  }
};

// FP64 kernel times: d=5 level 5, 1e4 points 15 us; d=30 level 3, 5e4 points
// 2,104 to 157 us; bound by the sums over the lanes and the LDS adds.
template <typename T, int DB, int K, bool kMod, int MD>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kMod ? 4 : 3)))
void tree_multT_kernel(const TreeMultTArgs a) {
  const int lane = threadIdx.x;
  const TreeChunk ch = a.chunks[blockIdx.x];
  double* acc = reinterpret_cast<double*>(tree_lds);
  for (int i = lane; i < ch.n; i += 64) acc[i] = 0.0;
  TreeScatter<T, K> sc;
  sc.part0 = ch.part0;
  sc.partn = ch.n;
  sc.lane = lane;
  const int64_t m0 = static_cast<int64_t>(blockIdx.y) * a.seg;
  const int64_t m1 = m0 + a.seg < a.mend ? m0 + a.seg : a.mend;
  for (int64_t mb = m0; mb < m1; mb += 64 * K) {
    const int64_t m = mb + lane;
    TreePoints<T, DB, K, kMod> pts;
    T y[K], all[K];
#pragma unroll
    for (int k = 0; k < K; ++k) y[k] = static_cast<const T*>(a.Y)[m + k * 64];
    pts.load(static_cast<const T*>(a.X), a.ldx, a.D, m, all);
    if (ch.root) {
      T c = T(0);
#pragma unroll
      for (int k = 0; k < K; ++k) c = fmaT(y[k], all[k], c);
      sc.add(0u, c);
    }
    if (ch.nrec > 0) {
      TreeWalk<T, DB, K, kMod, MD, TreeScatter<T, K>> walk{pts, sc, nullptr, TreeRecWords{}, a.D};
      walk.run((TreeRecPtr)(a.recs + ch.rec0), y);
    }
  }
  // (one wave: its LDS operations are in order)
  double* out = a.part + static_cast<int64_t>(blockIdx.y) * a.ntable + ch.off0;
  for (int i = lane; i < ch.n; i += 64) out[i] = acc[i];
}

template <typename T, int DB, int K, bool kMod, int MD>
void launch_tree_mult(const TreeMultArgs& a, dim3 grid, unsigned block, unsigned lds,
                      hipStream_t s) {
  clear_launch_error();
  hipLaunchKernelGGL((tree_mult_kernel<T, DB, K, kMod, MD>), grid, dim3(block), lds, s, a);
}
template <typename T, int DB, int K, bool kMod, int MD>
void launch_tree_multT(const TreeMultTArgs& a, dim3 grid, unsigned lds, hipStream_t s) {
  clear_launch_error();
  hipLaunchKernelGGL((tree_multT_kernel<T, DB, K, kMod, MD>), grid, dim3(64), lds, s, a);
}

// data points per lane of the wide variants
template <typename T>
constexpr int tree_k(int DB) {
  return sizeof(T) == 4 ? (DB <= 10 ? 4 : 2) : (DB <= 10 ? 2 : 1);
}

template <typename T, bool kMod, int DB>
TreeLaunch tree_variant(int depth, bool wide) {
  constexpr int K = tree_k<T>(DB == 0 ? 20 : DB);
  constexpr int kFew = DB == 4 ? 4 : 6;  // register sets of the usual variants
  TreeLaunch l;
  if (depth > kFew) {
    l.mult = &launch_tree_mult<T, DB, 1, kMod, kTreeMaxDepth>;
    l.multT = &launch_tree_multT<T, DB, 1, kMod, kTreeMaxDepth>;
  } else if (wide) {
    l.k = l.kt = K;
    l.mult = &launch_tree_mult<T, DB, K, kMod, kFew>;
    l.multT = &launch_tree_multT<T, DB, K, kMod, kFew>;
  } else {
    l.mult = &launch_tree_mult<T, DB, 1, kMod, kFew>;
    l.multT = &launch_tree_multT<T, DB, 1, kMod, kFew>;
  }
  return l;
}

}  // namespace

template <typename T, bool kMod>
TreeLaunch tree_launch(int D, int depth, bool wide) {
  if (depth > kTreeMaxDepth) throw device_error("tree deeper than the kernels' register sets");
  if (D <= 4) return tree_variant<T, kMod, 4>(depth, wide);
  if (D <= 8) return tree_variant<T, kMod, 8>(depth, wide);
  if (D <= 10) return tree_variant<T, kMod, 10>(depth, wide);
  if (D <= 16) return tree_variant<T, kMod, 16>(depth, wide);
  if (D <= 20) return tree_variant<T, kMod, 20>(depth, wide);
  return tree_variant<T, kMod, 0>(depth, wide);
}

}  // namespace sgpp_hip
