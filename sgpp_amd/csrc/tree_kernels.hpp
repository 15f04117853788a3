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

// one instruction: the C++ form adds a range check (2^32 gives 2^32 - 1)
__device__ __forceinline__ unsigned to_fixed(float x) {
  unsigned r;
  asm("v_cvt_u32_f32 %0, %1" : "=v"(r) : "v"(x));
  return r;
}
__device__ __forceinline__ unsigned to_fixed(double x) {
  unsigned r;
  asm("v_cvt_u32_f64 %0, %1" : "=v"(r) : "v"(x));
  return r;
}
// one instruction each (no canonicalisation): min(a, b), max(|a|, b)
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
__device__ __forceinline__ float max_abs(float a, float b) {
  float r;
  asm("v_max_f32 %0, |%1|, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_abs(double a, double b) {
  double r;
  asm("v_max_f64 %0, |%1|, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float rint_raw(float a) { return __builtin_rintf(a); }
__device__ __forceinline__ double rint_raw(double a) { return __builtin_rint(a); }
__device__ __forceinline__ float scale_of(uint32_t bits, float) { return __uint_as_float(bits); }
__device__ __forceinline__ double scale_of(uint32_t bits, double) {
  return __hiloint2double(static_cast<int>(bits), 0);
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

// Linear grids walked with the dimensions passed (kTreePassDims)
template <int DB, bool kMod>
constexpr bool kTreePass = !kMod && DB > 0 && DB <= kTreePassDims;

// The data points of a walk, as tree_points_kernel stores them: per dimension
// the coordinate times 2^32 and, for Linear grids, 2^D times the product of the later
// dimensions' halved level-1 factors (kTreePass) or 2 over the level-1 factor, in
// registers (DB > 0) or, for many dimensions (DB == 0), read from memory when a
// run begins; and the product of all level-1 factors.
template <typename T, int DB, int K, bool kMod>
struct TreePoints {
  DimRegs<T, DB> x[K], c[kMod ? 1 : K];
  __device__ __forceinline__ void load(const T* __restrict__ X, int64_t ldx, int D, int64_t m,
                                       T (&one)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) one[k] = kMod ? T(1) : X[2 * D * ldx + m + k * 64];
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const int from = min(d, D - 1);  // (the rest are not read; no branches)
#pragma unroll
      for (int k = 0; k < K; ++k) {
        x[k].set(d, X[from * ldx + m + k * 64]);
        if constexpr (!kMod) c[k].set(d, X[(D + from) * ldx + m + k * 64]);
      }
    }
  }
  __device__ __forceinline__ void coordinates(int r, T (&xr)[K]) const { dim_values(x, r, xr); }
  __device__ __forceinline__ void values(int r, T (&xr)[K], T (&cr)[K]) const {
    if constexpr (kMod) {
      coordinates(r, xr);
    } else {
      const DimRegs<T, DB>(*const v[2])[K] = {&x, &c};
      T(*const out[2])[K] = {&xr, &cr};
      dim_values<T, DB, K, 2>(v, r, out);
    }
  }
};
template <typename T, int K, bool kMod>
struct TreePoints<T, 0, K, kMod> {
  const T* p;
  int64_t ld;
  int dims;
  __device__ __forceinline__ void load(const T* __restrict__ X, int64_t ldx, int D, int64_t m,
                                       T (&one)[K]) {
    p = X + m;
    ld = ldx;
    dims = D;
#pragma unroll
    for (int k = 0; k < K; ++k) one[k] = kMod ? T(1) : p[2 * D * ldx + k * 64];
  }
  __device__ __forceinline__ void values(int r, T (&xr)[K], T (&cr)[K]) const {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      xr[k] = p[r * ld + k * 64];
      if constexpr (!kMod) cr[k] = p[(dims + r) * ld + k * 64];
    }
  }
};

// The walk over a chunk's program. Per depth the product R of all factors of
// the subspace at that depth (level 1 in the dimensions not refined) and its
// table position F. A run (the children of one parent in one dimension)
// fetches x 2^32, whose integer part's top l - 1 bits are the cell of level l,
// and rr, twice the product of all factors but the run's own. Per node and
// data point, with v = 2^(l-1) x (its cells are the unit intervals):
//   Linear: half the hat is |v - rint(v)|, the distance to the nearest cell
//     edge (exact). With kTreePass R is the product of the halved factors of the
//     dimensions up to the subspace's last refined one, extended at a run by those
//     it passes, and rr R times the product of the later ones (which holds the
//     halves' 2^D); otherwise R times 2 over the dimension's level-1 factor
//     takes that factor out.
//   ModLinear: level-1 factors are 1. The extrapolated boundary functions are
//     2 - 2^l min(x, 1-x), which exceeds the hat in the boundary cells only:
//     the larger of the two.
// A point on a cell edge may round to either side: the hat is 0 there.
template <typename T, int DB, int K, bool kMod, int MD, typename Use>
struct TreeWalk {
  TreePoints<T, DB, K, kMod>& pts;
  Use use;
  TreeRecPtr next;
  TreeRecWords cur;
  T xr[K], cr[K], rr[K];
  unsigned fx[K];

  __device__ __forceinline__ void run(TreeRecPtr recs, T (&R0)[K]) {
    next = recs;
    cur = next[0];
    unsigned F0[K];
#pragma unroll
    for (int k = 0; k < K; ++k) F0[k] = 0u;
    level<0>(R0, F0);
  }

  static constexpr bool kPass = kTreePass<DB, kMod>;
  template <int kDepth>
  __device__ __forceinline__ void level(T (&R)[K], const unsigned (&F)[K]) {
    for (;;) {
      const unsigned off = cur.x, ctl = cur.y, scale = cur.z;
      ++next;
      cur = next[0];  // in flight during this node
      if (ctl & kTreeRun) {
        const int r = (ctl >> kTreeDimShift) & 63u;
        if constexpr (kPass)
          for (int d = r - static_cast<int>((ctl >> kTreePassShift) & 15u); d < r; ++d) {
            T h[K];
            pts.coordinates(d, h);
#pragma unroll
            for (int k = 0; k < K; ++k)
              R[k] *= min_raw(h[k], T(4294967296.0) - h[k]) * T(0x1.0p-32);
          }
        pts.values(r, xr, cr);
#pragma unroll
        for (int k = 0; k < K; ++k) {
          fx[k] = to_fixed(xr[k]);
          if constexpr (kMod) cr[k] = min_raw(xr[k], T(4294967296.0) - xr[k]);
          rr[k] = kMod ? R[k] + R[k] : R[k] * cr[k];
        }
      }
      unsigned E[K];
#pragma unroll
      for (int k = 0; k < K; ++k) E[k] = __builtin_amdgcn_alignbit(F[k], fx[k], ctl);
      use.begin(off, ctl, E);
      const T L = scale_of(scale, T(0));
      T P[K], e[K];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const T v = xr[k] * L;
        e[k] = v - rint_raw(v);
        P[k] = rr[k] * (kMod ? max_abs(e[k], fmaT(-L, cr[k], T(1))) : absT(e[k]));
      }
      use.end(off, ctl, P, E);
      if (ctl & (kTreePush | kTreeLast | kTreeFlush)) {
        if (sizeof(T) == 4 && (ctl & kTreeFlush)) use.flush();
        if constexpr (kDepth + 1 < MD)
          if (ctl & kTreePush) {
            if constexpr (kPass) {
#pragma unroll
              for (int k = 0; k < K; ++k) P[k] = R[k] * absT(e[k]);
            }
            level<kDepth + 1>(P, E);
          }
        if (ctl & kTreeLast) return;
      }
    }
  }
};

extern __shared__ __align__(16) unsigned char tree_lds[];

// byte address in LDS (the kernels have no LDS but tree_lds, which begins at 0: their
// fixed size is tested. Adding tree_lds's address left an addition of 0 at every read)
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

// mult: bound by vector instructions, most of which issue every four cycles in
// either precision: seven (Linear) or nine per node and data point, four per run and
// five per dimension passed (one scalar instruction issues in four cycles, so several
// points per lane share a node's). The weights of a chunk's subspaces are gathered from LDS, where up to
// 64 cells meet no bank conflict. Kernel times against the culled kernels: Linear
// d=8 level 6, 5e5 points, FP32 1,179 to 260 us, FP64 1,678 to 403; d=20 adaptive,
// 5e5 points, FP32 6,523 to 3,023; ModLinear d=10 adaptive, 1e6 points, FP32 2,051
// to 1,403. Taking level-1 factors out, instead of passing dimensions: d=20 4,960 to
// 3,020 us; d=8 260 to 230, but with a larger error than the culled kernels'
// (kTreePassDims).
template <typename T, int DB, int K, bool kMod, int MD>
__global__ __launch_bounds__(kTreeBlock) __attribute__((amdgpu_waves_per_eu(kMod ? 4 : 3)))
void tree_mult_kernel(const TreeMultArgs a) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t m = static_cast<int64_t>(blockIdx.x) * blockDim.x * K + wave * 64 * K + lane;
  T* lds = reinterpret_cast<T*>(tree_lds);
  TreePoints<T, DB, K, kMod> pts;
  T all[K];
  pts.load(static_cast<const T*>(a.X), a.ldx, a.D, m, all);
  TreeGather<T, K> g;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    g.acc[k] = T(0);
    g.accd[k] = 0.0;
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
      for (int k = 0; k < K; ++k) g.accd[k] += static_cast<double>(w * all[k]);
    }
    if (ch.nrec > 0) {
      TreeWalk<T, DB, K, kMod, MD, TreeGather<T, K>> walk{pts, g, nullptr, TreeRecWords{}};
      T start[K];
#pragma unroll
      for (int k = 0; k < K; ++k) start[k] = kTreePass<DB, kMod> ? T(1) : all[k];
      walk.run((TreeRecPtr)(a.recs + ch.rec0), start);
      g = walk.use;
      g.flush();
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const double r = g.accd[k];
    const int64_t row = m + k * 64;
    if (a.part)
      a.part[static_cast<int64_t>(blockIdx.y) * a.ldx + row] = r;
    else if (const int32_t j = a.sperm[row]; j >= 0)
      a.out[j] = r;
  }
}

// v with all bits kept or cleared
__device__ __forceinline__ float and_bits(float v, unsigned m) {
  return __uint_as_float(__float_as_uint(v) & m);
}
__device__ __forceinline__ double and_bits(double v, unsigned m) {
  return __hiloint2double(static_cast<int>(static_cast<unsigned>(__double2hiint(v)) & m),
                          static_cast<int>(static_cast<unsigned>(__double2loint(v)) & m));
}

// multTranspose: each data point's value is added to its table position, in
// LDS, in FP64. Equal positions in one LDS add wait for each other (64 equal
// ones 192 cycles, 64 different ones 9), so values are joined first: the points
// of a pair of lanes are consecutive in storage order (tree_points_kernel) and
// mostly in one position; the pairs are far apart. Joining two or three steps more
// cost more instructions than the conflicts they saved (d=8 level 6, FP64:
// 706 and 767 us against 675), none at all cost 667 against 598 later.
template <typename T, int K>
struct TreeScatter {
  unsigned part0, partn;
  unsigned keep;  // all ones in the lane of a pair that keeps the joined value
  __device__ __forceinline__ void begin(uint32_t, uint32_t, const unsigned (&)[K]) {}
  __device__ __forceinline__ void flush() {}
  __device__ __forceinline__ void add(unsigned byte, T c) {
    atomicAdd(reinterpret_cast<double*>(tree_lds + byte), static_cast<double>(c));
  }
  __device__ __forceinline__ void end(uint32_t off, uint32_t ctl, const T (&P)[K],
                                      const unsigned (&E)[K]) {
    if (ctl & kTreeTable) {
      T v[K];
#pragma unroll
      for (int k = 0; k < K; ++k) v[k] = P[k];
#pragma unroll
      for (int w = 1; w < K; w *= 2)
#pragma unroll
        for (int k = 0; k + w < K; k += 2 * w) {
          const bool differ = E[k] != E[k + w];
          T c = differ ? T(0) : v[k + w];
          asm("" : "+v"(c));  // (a select, not a branch)
          if (__ballot(differ) != 0ull)
            if (differ) add(off + E[k + w] * 8u, v[k + w]);
          v[k] += c;
        }
      static_assert(kTreeJoin == 1, "lanes join in pairs");
      constexpr int kPair = 0xb1;  // quad_perm [1,0,3,2]
      const unsigned e = static_cast<unsigned>(
          __builtin_amdgcn_mov_dpp(static_cast<int>(E[0]), kPair, 0xf, 0xf, true));
      const T sum = and_bits(v[0] + dpp_z<kPair>(v[0]), keep);
      v[0] = E[0] == e ? sum : v[0];
      if (v[0] != T(0)) add(off + E[0] * 8u, v[0]);
    } else if (ctl & kTreePart) {
#pragma unroll
      for (int k = 0; k < K; ++k)
        if (E[k] - part0 < partn) add(off + E[k] * 8u, P[k]);
    }
  }
};

// Waves per SIMD: three where four (128 registers) spill the coordinates and
// products of several points. Kernel times with four and three, level 5, 3e5
// points: d=10 FP32 651 and 248 us, FP64 563 and 334; d=8 level 6, 5e5 points, FP32
// 515 and 451; FP64 there spills two registers only, 579 and 648.
template <typename T, int DB, int K, bool kMod>
constexpr int tree_multT_waves() {
  return kTreePass<DB, kMod> && K > 1 && DB >= (sizeof(T) == 4 ? 8 : 10) ? 3 : 4;
}

// Bound by vector instructions, the LDS adds about half of the time beside them.
// Kernel times against the culled kernel: Linear d=8 level 6, 5e5 points, FP32
// 1,621 to 451 us, FP64 2,300 to 579; ModLinear d=10 adaptive, 1e6 points, FP32
// 2,218 to 1,903; against the subspace algorithm's own, d=7 level 6, 2.5e5 points,
// 681 to 224 with the final sums.
template <typename T, int DB, int K, bool kMod, int MD>
__global__ __launch_bounds__(64)
__attribute__((amdgpu_waves_per_eu(tree_multT_waves<T, DB, K, kMod>())))
void tree_multT_kernel(const TreeMultTArgs a) {
  const int lane = threadIdx.x;
  const TreeItem it = a.items[blockIdx.x];
  const TreeChunk ch = a.chunks[it.chunk];
  double* acc = reinterpret_cast<double*>(tree_lds);
  for (int i = lane; i < ch.n; i += 64) acc[i] = 0.0;
  __syncthreads();  // (one wave, whose LDS operations are in order: for the compiler)
  TreeScatter<T, K> sc;
  sc.part0 = ch.part0;
  sc.partn = ch.n;
  sc.keep = lane & 1 ? 0u : ~0u;
  for (int b = it.b0; b < it.b1; ++b) {
    const int64_t m = static_cast<int64_t>(b) * (64 * K) + lane;
    TreePoints<T, DB, K, kMod> pts;
    T y[K], all[K];
#pragma unroll
    for (int k = 0; k < K; ++k) y[k] = static_cast<const T*>(a.Y)[m + k * 64];
    pts.load(static_cast<const T*>(a.X), a.ldx, a.D, m, all);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      all[k] *= y[k];
      if constexpr (!kTreePass<DB, kMod>) y[k] = all[k];
    }
    if (ch.root) {
      T c = T(0);
#pragma unroll
      for (int k = 0; k < K; ++k) c += all[k];
      c = sum_to_lane63(c);
      if (lane == 63) sc.add(0u, c);
    }
    if (ch.nrec > 0) {
      TreeWalk<T, DB, K, kMod, MD, TreeScatter<T, K>> walk{pts, sc, nullptr, TreeRecWords{}};
      walk.run((TreeRecPtr)(a.recs + ch.rec0), y);
    }
  }
  __syncthreads();
  double* out = a.part + it.off;
  for (int i = lane; i < ch.n; i += 64) out[i] = acc[i];
}

template <typename T, int DB, int K, bool kMod, int MD>
void launch_tree_mult(const TreeMultArgs& a, dim3 grid, unsigned block, unsigned lds,
                      hipStream_t s) {
  clear_launch_error();
  hipLaunchKernelGGL((tree_mult_kernel<T, DB, K, kMod, MD>), grid, dim3(block), lds, s, a);
}
template <typename T, int DB, int K, bool kMod, int MD>
void launch_tree_multT(const TreeMultTArgs& a, unsigned items, unsigned lds, hipStream_t s) {
  clear_launch_error();
  hipLaunchKernelGGL((tree_multT_kernel<T, DB, K, kMod, MD>), dim3(items), dim3(64), lds, s, a);
}

// data points per lane of the wide variants
template <typename T>
constexpr int tree_k(int DB) {
  return sizeof(T) == 4 ? (DB <= 10 ? 4 : 2) : (DB <= 10 ? 2 : 1);
}

template <typename T, bool kMod, int DB>
TreeLaunch tree_variant(int depth, bool wide) {
  constexpr int K = tree_k<T>(DB == 0 ? 20 : DB);
  constexpr int kFew = tree_few_dims(DB == 0 ? 64 : DB);  // register sets of the usual variants
  TreeLaunch l;
  if (depth > kFew) {
    l.mult = &launch_tree_mult<T, DB, 1, kMod, kTreeMaxDepth>;
    l.multT = &launch_tree_multT<T, DB, 1, kMod, kTreeMaxDepth>;
  } else if (wide) {
    l.k = K;
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
