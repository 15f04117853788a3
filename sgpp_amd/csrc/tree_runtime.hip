// Runtime of the subspace-tree algorithm (tree_device.hpp): grids and
// programs on the host, launch shapes, the small kernels around the walks.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "parts_device.hpp"
#include "tree_device.hpp"

namespace sgpp_hip {

namespace {

// W[e] = alpha[ti[e]] in the compute type (0 where the entry has no grid point)
template <typename T>
__global__ void tree_weights_kernel(const double* __restrict__ alpha,
                                    const int32_t* __restrict__ ti, T* __restrict__ W, int64_t n) {
  const int64_t e = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (e < n) W[e] = ti[e] >= 0 ? static_cast<T>(alpha[ti[e]]) : T(0);
}

// a product in two doubles (one rounding in the end instead of one a factor)
struct Product {
  double hi = 1.0, lo = 0.0;
  __device__ __forceinline__ void times(double f) {
    const double p = hi * f;
    lo = fma(hi, f, -p) + lo * f;
    hi = p;
  }
  __device__ __forceinline__ double value() const { return hi + lo; }
};

// The data as the walks read them, in batches of 64 K rows (row 64 k + l of a
// batch is lane l's point k): the lanes that multTranspose joins have consecutive
// stored rows, and such groups are spread evenly over all rows. X: [D][ldx]. XT: per
// dimension a row of 2^32 x; for Linear grids then per dimension a row of 2^D times
// the product of the later dimensions' halved level-1 factors (D <= kTreePassDims)
// or of 2 over the level-1 factor, and a row of the products of the level-1 factors.
// Rows past M are copies of row M - 1 whose caller's row sperm is -1.
template <typename T, bool kMod>
__global__ void tree_points_kernel(const T* __restrict__ X, int64_t ldx,
                                   const int32_t* __restrict__ dperm, int64_t M, int D, int K,
                                   int64_t rows, T* __restrict__ XT,
                                   int32_t* __restrict__ sperm) {
  // (below this the reciprocal of a halved level-1 factor could overflow)
  constexpr double kTiny = sizeof(T) == 4 ? 0x1.0p-127 : 0x1.0p-1023;
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  constexpr int kGroup = 1 << kTreeJoin, kGroups = 64 / kGroup;
  const int lane = r % 64, k = r / 64 % K;
  const int64_t m = (lane / kGroup) * (rows / kGroups) + r / (64 * K) * (kGroup * K) +
                    (lane % kGroup) * K + k;
  const int64_t from = m < M ? m : M - 1;
  sperm[r] = m < M ? dperm[m] : -1;
  const bool pass = D <= kTreePassDims;
  Product all;
  all.hi = ldexp(1.0, D);
  for (int d = D - 1; d >= 0; --d) {
    const double x = static_cast<double>(X[d * ldx + from]);
    XT[d * rows + r] = static_cast<T>(x * 0x1.0p32);
    if (kMod) continue;
    double half = fmin(x, 1.0 - x);
    if (pass) {
      XT[(D + d) * rows + r] = static_cast<T>(all.value());
    } else {
      if (half < kTiny) half = 0.0;
      XT[(D + d) * rows + r] = static_cast<T>(half == 0.0 ? 0.0 : 1.0 / half);
    }
    all.times(half);
  }
  if (!kMod) XT[2 * D * rows + r] = static_cast<T>(all.value());
}

// Y[r] = y[sperm[r]], 0 where sperm is -1
template <typename T>
__global__ void tree_prep_kernel(const double* __restrict__ y, const int32_t* __restrict__ sperm,
                                 T* __restrict__ Y, int64_t n) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (r < n) Y[r] = sperm[r] >= 0 ? static_cast<T>(y[sperm[r]]) : T(0);
}

// out[ti[e]] = the sum of a table entry's partial sums, rows added in a fixed order
__global__ __launch_bounds__(kRows* kCols) void tree_sum_kernel(
    const double* __restrict__ part, const TreeSum* __restrict__ sums,
    const int32_t* __restrict__ ti, double* __restrict__ out) {
  const TreeSum q = sums[blockIdx.x];
  const int c = threadIdx.x % kCols;
  const double s = sum_rows(part + q.off + c, q.ld, c < q.n ? q.rows : 0);
  if (threadIdx.x >= kCols || c >= q.n) return;
  const int32_t j = ti[q.e0 + c];
  if (j >= 0) out[j] = s;
}

}  // namespace

namespace {

// The steps of a level vector, (dimension, level above 1) one by one: five of 12 bits
// in a word, the first at the top, 0 where there is none. So keys compare as the
// depth-first order does, a parent before its children.
constexpr int kStepsPerWord = 5;
template <int W>
struct StepKey {
  uint64_t w[W];
  uint32_t j;
  bool same(const StepKey& o) const { return std::equal(w, w + W, o.w); }
};

template <int W>
bool tree_nodes(size_t D, size_t N, const uint32_t* level, TreeGrid& g) {
  std::vector<StepKey<W>> key(N);
  for (size_t j = 0; j < N; ++j) {
    StepKey<W>& k = key[j];
    k = StepKey<W>{};
    k.j = static_cast<uint32_t>(j);
    int n = 0;
    for (size_t d = 0; d < D; ++d)
      if (const uint64_t l = level[j * D + d]; l > 1) {
        k.w[n / kStepsPerWord] |= ((d + 1) << 5 | l) << (12 * (kStepsPerWord - 1 - n % kStepsPerWord));
        ++n;
      }
  }
  std::sort(key.begin(), key.end(), [](const StepKey<W>& x, const StepKey<W>& y) {
    for (int i = 0; i < W; ++i)
      if (x.w[i] != y.w[i]) return x.w[i] < y.w[i];
    return x.j < y.j;
  });
  const int64_t limit = subspace_table_limit(N);
  g.order.resize(N);
  for (size_t s = 0; s < N; ++s) {
    g.order[s] = key[s].j;
    if (s && key[s].same(key[s - 1])) continue;
    TreeGrid::Node n{0, g.total, 0};
    const uint32_t* lv = level + static_cast<size_t>(key[s].j) * D;
    int64_t bits = 0;
    for (size_t d = 0; d < D; ++d) {
      n.depth += lv[d] > 1;
      bits += lv[d] - 1;
      g.level.push_back(static_cast<uint8_t>(lv[d]));
    }
    if (bits > 30) return false;
    n.bits = static_cast<int>(bits);
    g.total += int64_t(1) << bits;
    if (g.total > limit) return false;
    g.node.push_back(n);
    g.first.push_back(static_cast<uint32_t>(s));
  }
  g.first.push_back(static_cast<uint32_t>(N));
  return true;
}

}  // namespace

bool build_tree_grid(size_t D, size_t N, const uint32_t* level, TreeGrid& g) {
  g = TreeGrid();
  g.D = D;
  for (size_t j = 0; j < N; ++j) {
    int n = 0;
    for (size_t d = 0; d < D; ++d) n += level[j * D + d] > 1;
    g.depth = std::max(g.depth, n);
  }
  if (g.depth > kTreeMaxDepth) return false;
  static_assert(kTreeMaxDepth <= 3 * kStepsPerWord, "a key holds every step");
  if (g.depth <= kStepsPerWord) return tree_nodes<1>(D, N, level, g);
  if (g.depth <= 2 * kStepsPerWord) return tree_nodes<2>(D, N, level, g);
  return tree_nodes<3>(D, N, level, g);
}

bool tree_tables(const TreeGrid& g, const uint32_t* level, const uint32_t* index,
                 std::vector<int32_t>& ti) {
  ti.assign(static_cast<size_t>(g.total), -1);
  for (size_t q = 0; q < g.node.size(); ++q)
    for (uint32_t s = g.first[q]; s < g.first[q + 1]; ++s) {
      const size_t j = g.order[s];
      int64_t flat = 0;
      for (size_t d = 0; d < g.D; ++d)
        if (const uint32_t l = level[j * g.D + d]; l > 1)
          flat = (flat << (l - 1)) + (index[j * g.D + d] >> 1);
      int32_t& entry = ti[static_cast<size_t>(g.node[q].off + flat)];
      if (entry >= 0) return false;
      entry = static_cast<int32_t>(j);
    }
  return true;
}

namespace {

// nodes between two additions of the FP32 sums to the FP64 ones
constexpr int kFlushNodes = 64;

struct Step {
  int dim, level;
};

// Appends the program of nodes [a, b) (b > a; the root, where it is one of
// them, is not a record). Table offsets are relative to off0; no_table: the
// nodes' tables are left to the caller's part chunk (kTreePart).
void append_program(const TreeGrid& g, size_t a, size_t b, int64_t off0, int entry_bytes, bool fp32,
                    bool part, TreeProgram& p) {  // (depth at most kTreeMaxDepth)
  struct Emit {
    int depth, dim, level;
    uint32_t off, flags;
  };
  std::vector<Emit> out;
  std::vector<Step> path, steps;
  int since = 0;
  for (size_t s = a; s < b; ++s) {
    const uint8_t* lv = &g.level[s * g.D];
    steps.clear();
    for (size_t d = 0; d < g.D; ++d)
      if (lv[d] > 1) steps.push_back(Step{static_cast<int>(d), lv[d]});
    if (steps.empty()) continue;  // the root
    size_t same = 0;
    while (same < path.size() && same < steps.size() && path[same].dim == steps[same].dim &&
           path[same].level == steps[same].level)
      ++same;
    // ancestors that are not on the path (at a chunk's start, or not in the
    // grid) are walked without a table
    for (size_t q = same; q + 1 < steps.size(); ++q)
      out.push_back(Emit{static_cast<int>(q), steps[q].dim, steps[q].level, 0u, 0u});
    uint32_t flags = part ? kTreePart : kTreeTable;
    if (fp32 && ++since == kFlushNodes) {
      flags |= kTreeFlush;
      since = 0;
    }
    out.push_back(Emit{static_cast<int>(steps.size()) - 1, steps.back().dim, steps.back().level,
                       static_cast<uint32_t>((part ? -off0 : g.node[s].off - off0) * entry_bytes),
                       flags});
    path = steps;
  }
  int passed[kTreeMaxDepth] = {};  // per depth: the dimensions before this one are passed
  for (size_t i = 0; i < out.size(); ++i) {
    Emit& e = out[i];
    if (i + 1 < out.size() && out[i + 1].depth == e.depth + 1) e.flags |= kTreePush;
    const bool follows = i > 0 && out[i - 1].depth == e.depth && out[i - 1].dim == e.dim &&
                         !(out[i - 1].flags & kTreePush);
    if (!follows) e.flags |= kTreeRun;
    size_t q = i + 1;
    while (q < out.size() && out[q].depth > e.depth) ++q;
    if (q == out.size() || out[q].depth < e.depth) e.flags |= kTreeLast;
    TreeRec r{};
    r.off = e.off;
    r.ctl = static_cast<uint32_t>(33 - e.level) | (static_cast<uint32_t>(e.dim) << kTreeDimShift) |
            e.flags;
    r.scale = fp32 ? static_cast<uint32_t>(127 + e.level - 33) << 23
                   : static_cast<uint32_t>(1023 + e.level - 33) << 20;
    if (g.D <= kTreePassDims) {
      // from the parent's dimension, or the run before, to this record's
      if (i == 0 || out[i - 1].depth < e.depth)
        passed[e.depth] = e.depth > 0 ? out[i - 1].dim + 1 : 0;
      r.ctl |= static_cast<uint32_t>(e.dim - passed[e.depth]) << kTreePassShift;
      passed[e.depth] = e.dim;
    }
    p.recs.push_back(r);
  }
}

}  // namespace

TreeProgram build_tree_program(const TreeGrid& g, int ngroups, int64_t cap, int64_t max_nodes,
                               int entry_bytes, bool fp32) {
  TreeProgram p;
  const size_t n = g.node.size();
  ngroups = static_cast<int>(std::max<size_t>(1, std::min<size_t>(ngroups, n)));
  for (int q = 0; q < ngroups; ++q) {
    const size_t g0 = n * q / ngroups, g1 = n * (q + 1) / ngroups;
    p.groups.push_back(static_cast<int>(p.chunks.size()));
    for (size_t a = g0; a < g1;) {
      const int64_t size = int64_t(1) << g.node[a].bits;
      if (size > cap) {
        // one subspace in parts of cap positions
        for (int64_t s = 0; s < size; s += cap) {
          TreeChunk c{};
          c.rec0 = static_cast<int>(p.recs.size());
          append_program(g, a, a + 1, s, entry_bytes, fp32, true, p);
          c.nrec = static_cast<int>(p.recs.size()) - c.rec0;
          c.n = static_cast<int>(std::min(cap, size - s));
          c.part0 = static_cast<int>(s);
          c.off0 = g.node[a].off + s;
          p.max_entries = std::max(p.max_entries, c.n);
          p.chunks.push_back(c);
        }
        ++a;
        continue;
      }
      size_t b = a;
      const int64_t off0 = g.node[a].off;
      int64_t entries = 0;
      while (b < g1 && static_cast<int64_t>(b - a) < max_nodes) {
        const int64_t more = int64_t(1) << g.node[b].bits;
        if (entries + more > cap) break;
        entries += more;
        ++b;
      }
      TreeChunk c{};
      c.rec0 = static_cast<int>(p.recs.size());
      append_program(g, a, b, off0, entry_bytes, fp32, false, p);
      c.nrec = static_cast<int>(p.recs.size()) - c.rec0;
      c.n = static_cast<int>(entries);
      c.off0 = off0;
      c.root = g.node[a].depth == 0;
      p.max_entries = std::max(p.max_entries, c.n);
      p.chunks.push_back(c);
      a = b;
    }
  }
  p.groups.push_back(static_cast<int>(p.chunks.size()));
  p.recs.push_back(TreeRec{});  // read ahead of the last record
  return p;
}

// ----------------------------------------------------------------- shapes

namespace {

// LDS of a mult block and of a multTranspose wave: 40 KiB and 10 KiB let the
// the registers bound the waves in flight (16 per CU, 12 for Linear)
constexpr int kMultLds = 40 << 10;
constexpr int kMultTEntries = 1280;
// nodes per chunk group (mult) or chunk (multTranspose) at least, so that a
// wave's start is small against its walk
constexpr int kMinNodes = 8;
// multTranspose: nodes times batches of a wave, and what a batch's loads cost in
// nodes
// (a d=8 regular grid, M=5e5: 2 rounds; a d=10 adaptive one, M=1e6: 2 rounds 2,058
// us with the final sums, 4 1,949, 16 1,943)
constexpr int64_t kMultTWork = 300;
constexpr int kBatchNodes = 5;
constexpr int64_t kTreePartialBudget = int64_t(2048) << 20;

}  // namespace

int64_t tree_walks(const TreeGrid& g, bool multT) {
  const int64_t cap = multT ? kMultTEntries : kMultLds / 8;
  int64_t n = 0;
  for (const TreeGrid::Node& q : g.node) {
    const int64_t size = int64_t(1) << q.bits;
    n += size > cap ? (size + cap - 1) / cap * q.depth : 1;
  }
  return n;
}

void DeviceMultiEval::upload_tree(const TreeProgram& p, TreePlan& plan, int entry_bytes) {
  plan.ngroups = static_cast<int>(p.groups.size()) - 1;
  plan.factors = static_cast<int64_t>(p.recs.size()) - 1;
  plan.lookups = 0;
  for (const TreeRec& r : p.recs) plan.lookups += (r.ctl & (kTreeTable | kTreePart)) != 0;
  for (const TreeChunk& c : p.chunks) plan.lookups += c.root;
  plan.lds = (p.max_entries * entry_bytes + 15) / 16 * 16;
  ensure(&plan.recs, &plan.recs_cap, p.recs.size() * sizeof(TreeRec));
  check_hip(hipMemcpy(plan.recs, p.recs.data(), p.recs.size() * sizeof(TreeRec),
                      hipMemcpyHostToDevice),
            "upload tree records");
  ensure(&plan.chunks, &plan.chunks_cap, p.chunks.size() * sizeof(TreeChunk));
  check_hip(hipMemcpy(plan.chunks, p.chunks.data(), p.chunks.size() * sizeof(TreeChunk),
                      hipMemcpyHostToDevice),
            "upload tree chunks");
  ensure(&plan.groups, &plan.groups_cap, p.groups.size() * sizeof(int));
  check_hip(hipMemcpy(plan.groups, p.groups.data(), p.groups.size() * sizeof(int),
                      hipMemcpyHostToDevice),
            "upload tree groups");
}

namespace {

template <typename T>
TreeLaunch tree_variant_of(bool mod, size_t D, int depth, bool wide) {
  return mod ? tree_launch<T, true>(static_cast<int>(D), depth, wide)
             : tree_launch<T, false>(static_cast<int>(D), depth, wide);
}

// waves that the registers let a CU have in flight
constexpr int64_t waves_per_cu(bool mod) { return mod ? 16 : 12; }

}  // namespace

// several points per lane where that leaves every wave slot a walk of kMinNodes
template <typename T>
bool DeviceMultiEval::tree_wide(const TreeGrid& g) const {
  const bool mod = basis_ == Basis::ModLinear;
  return static_cast<int64_t>(M_) * static_cast<int64_t>(g.node.size()) >=
         num_cus_ * waves_per_cu(mod) * 64 * tree_variant_of<T>(mod, D_, g.depth, true).k * kMinNodes;
}

// The walks' times, fitted to the same pairs as own_times(): a launch or three; per
// data point and node (parts of a table are walked each, with adds that meet in
// multTranspose; walks of more than tree_few_dims() refined dimensions take one
// point per lane, those of more than kRegDims dimensions read them from memory) and per
// data point; what a block of mult copies of the tables, and the chain of one table's
// parts; multTranspose's partial sums and the rows that a final sum adds.
DeviceMultiEval::PathTimes DeviceMultiEval::tree_times(const TreeGrid& g) const {
  constexpr size_t kRegDims = 20;  // (of tree_launch)
  // 1e-6 us per data point and node, mult and multTranspose: up to 10 dimensions
  // (Linear, ModLinear), more, deep, more than kRegDims; per data point (multTranspose)
  constexpr double kNode[2][5][2] = {
      {{0.55, 1.11}, {0.51, 0.83}, {0.73, 1.28}, {0.8, 1.45}, {1.25, 2.0}},
      {{0.33, 0.6}, {0.345, 0.52}, {0.4, 0.7}, {0.76, 1.24}, {0.9, 1.4}}};
  constexpr double kPoint[5] = {30.0, 30.0, 100.0, 35.0, 50.0};
  const bool fp32 = serves(Precision::FP32), mod = basis_ == Basis::ModLinear;
  const bool wide = fp32 ? tree_wide<float>(g) : tree_wide<double>(g);
  const TreeLaunch l = fp32 ? tree_variant_of<float>(mod, D_, g.depth, wide)
                            : tree_variant_of<double>(mod, D_, g.depth, wide);
  const int c = D_ > kRegDims ? 4 : (g.depth > tree_few_dims(D_) ? 3 : (D_ > 10 ? 2 : mod));
  const double M = static_cast<double>(M_), nodes = static_cast<double>(g.node.size()),
               total = static_cast<double>(g.total),
               walks = static_cast<double>(tree_walks(g, false)),
               walksT = static_cast<double>(tree_walks(g, true));
  const double blocks = std::ceil(M / (kTreeBlock * l.k));
  const double rows = std::min(M / (64 * l.k), 24576.0 / std::max(1.0, total / kMultTEntries));
  return {20.0 + 1e-6 * (kNode[fp32][c][0] * walks + 8.0) * M + 1.2e-6 * total * blocks +
              50e-6 * total + 0.25 * (walks - nodes),
          26.0 + 1e-6 * (kNode[fp32][c][1] * (2.0 * walksT - nodes) + kPoint[c]) * M +
              25e-6 * total + 0.015 * rows};
}

template <typename T>
void DeviceMultiEval::set_tree_plans(const TreeGrid& g, bool mult, bool multT) {
  const int ix = sizeof(T) == sizeof(double) ? 0 : 1;
  const bool mod = basis_ == Basis::ModLinear;
  const int64_t nodes = static_cast<int64_t>(g.node.size());
  const int64_t M = static_cast<int64_t>(M_);
  const int64_t slots = num_cus_ * waves_per_cu(mod);
  tree_wide_[ix] = tree_wide<T>(g);
  const TreeLaunch l = tree_variant_of<T>(mod, D_, g.depth, tree_wide_[ix]);
  // the data in the walks' order
  const int64_t rb = (M + kTreeBlock * l.k - 1) / (kTreeBlock * l.k);
  const int64_t rows = tree_rows_[ix] = rb * kTreeBlock * l.k;
  ensure(&tree_x_[ix], &tree_x_cap_[ix], (mod ? D_ : 2 * D_ + 1) * rows * sizeof(T));
  ensure(&tree_sperm_[ix], &tree_sperm_cap_[ix], rows * sizeof(int32_t));
  clear_launch_error();
  hipLaunchKernelGGL((mod ? tree_points_kernel<T, true> : tree_points_kernel<T, false>),
                     dim3(blocks(rows, 256)), dim3(256), 0, stream_,
                     static_cast<const T*>(sizeof(T) == sizeof(double) ? X64_ : X32_),
                     static_cast<int64_t>(Mpad_), static_cast<const int32_t*>(dperm_), M,
                     static_cast<int>(D_), l.k, rows, static_cast<T*>(tree_x_[ix]),
                     static_cast<int32_t*>(tree_sperm_[ix]));
  check_hip(hipGetLastError(), "tree data order");
  if (mult) set_tree_mult<T>(g, rb, slots);
  if (multT) set_tree_multT<T>(g, rows / (64 * l.k));
}

// mult: chunk groups so that the blocks (rb per group) fill the slots evenly
template <typename T>
void DeviceMultiEval::set_tree_mult(const TreeGrid& g, int64_t rb, int64_t slots) {
  TreePlan& pm = tree_mult_[sizeof(T) == sizeof(double) ? 0 : 1];
  const int64_t nodes = static_cast<int64_t>(g.node.size());
  const int64_t bslots = slots / (kTreeBlock / 64);
  const int64_t gmax = std::max<int64_t>(1, nodes / kMinNodes);
  int64_t G = cfg_.mult_grid_chunks;
  if (G <= 0 && cfg_.target_blocks > 0) {
    G = std::min(gmax, (cfg_.target_blocks + rb - 1) / rb);
  } else if (G <= 0) {
    double best = 0.0;
    for (int64_t q = 1; q <= std::min<int64_t>(64, gmax); ++q) {
      // nanoseconds per data point: the walk with the last round's idle
      // blocks, the FP64 partials written and read
      const double b = static_cast<double>(rb * q);
      const double walk = 2e-4 * static_cast<double>(nodes) *
                          std::ceil(b / static_cast<double>(bslots)) * static_cast<double>(bslots) / b;
      const double t = walk + (q > 1 ? 0.005 * static_cast<double>(q) : 0.0);
      if (q == 1 || t < best * 0.98) {
        best = t;
        G = q;
      }
    }
  }
  // (also where the caller sets G: the subspace algorithm's own kernels had no partials)
  G = std::min<int64_t>(G, std::max<int64_t>(1, kTreePartialBudget / (Mpad_ * sizeof(double))));
  upload_tree(build_tree_program(g, static_cast<int>(std::min<int64_t>({G, nodes, 65535})),
                                 (kMultLds - 16) / static_cast<int64_t>(sizeof(T)), nodes,
                                 static_cast<int>(sizeof(T)), sizeof(T) == 4),
              pm, static_cast<int>(sizeof(T)));
}

// multTranspose: chunks; each a wave per data segment, the segments of a chunk
// by its nodes, so that all waves take about as long (with as many segments for
// every chunk, 44 % of the wave slots stood idle on a d=10 adaptive grid:
// 3,030 us against 1,900)
template <typename T>
void DeviceMultiEval::set_tree_multT(const TreeGrid& g, int64_t batches) {
  TreePlan& pt = tree_multT_[sizeof(T) == sizeof(double) ? 0 : 1];
  const int64_t nodes = static_cast<int64_t>(g.node.size());
  const int64_t tslots = static_cast<int64_t>(num_cus_) * 16;
  const int64_t rounds = std::max<int64_t>(
      2, std::min<int64_t>(6, nodes * batches / (kMultTWork * tslots)));
  const int64_t per = std::max<int64_t>(kMinNodes, nodes * batches / tslots);
  const TreeProgram p = build_tree_program(g, 1, kMultTEntries, per, 8, sizeof(T) == 4);
  upload_tree(p, pt, 8);
  const double target = cfg_.target_blocks > 0 ? cfg_.target_blocks
                                               : static_cast<double>(tslots * rounds);
  const double budget = static_cast<double>(kTreePartialBudget / 8) / static_cast<double>(g.total);
  double work = 0.0;
  for (const TreeChunk& c : p.chunks) work += c.nrec + kBatchNodes;
  std::vector<TreeItem> items;
  std::vector<TreeSum> sums;
  int64_t off = 0;
  pt.segs = 1;
  for (size_t c = 0; c < p.chunks.size(); ++c) {
    const TreeChunk& ch = p.chunks[c];
    const double asked = cfg_.multT_data_segs > 0 ? cfg_.multT_data_segs
                                                  : target * (ch.nrec + kBatchNodes) / work + 0.5;
    int64_t S = static_cast<int64_t>(std::min(budget, asked));
    S = std::max<int64_t>(1, std::min<int64_t>(S, batches));
    const int64_t len = (batches + S - 1) / S;
    S = (batches + len - 1) / len;
    pt.segs = std::max<int>(pt.segs, static_cast<int>(S));
    for (int i = 0; i < ch.n; i += kCols)
      sums.push_back(TreeSum{std::min(kCols, ch.n - i), static_cast<int>(S), off + i, ch.n,
                             ch.off0 + i});
    for (int64_t s = 0; s < S; ++s, off += ch.n)
      items.push_back(TreeItem{static_cast<int>(c), static_cast<int>(s * len),
                               static_cast<int>(std::min(batches, (s + 1) * len)), 0, off, 0});
  }
  pt.part = static_cast<size_t>(off) * sizeof(double);
  pt.nitems = static_cast<int>(items.size());
  pt.nsums = static_cast<int>(sums.size());
  ensure(&pt.items, &pt.items_cap, items.size() * sizeof(TreeItem));
  check_hip(hipMemcpy(pt.items, items.data(), items.size() * sizeof(TreeItem),
                      hipMemcpyHostToDevice),
            "upload tree items");
  ensure(&pt.sums, &pt.sums_cap, sums.size() * sizeof(TreeSum));
  check_hip(hipMemcpy(pt.sums, sums.data(), sums.size() * sizeof(TreeSum), hipMemcpyHostToDevice),
            "upload tree sums");
}

bool DeviceMultiEval::set_tree(const TreeGrid& g, const uint32_t* level, const uint32_t* index,
                               bool mult, bool multT) {
  std::vector<int32_t> ti;
  if (g.node.size() > (size_t(1) << 24) || !tree_tables(g, level, index, ti)) return false;
  check_hip(hipSetDevice(device_), "hipSetDevice");
  check_hip(hipStreamSynchronize(stream_), "hipStreamSynchronize");
  ensure(&tree_ti_, &tree_ti_cap_, ti.size() * sizeof(int32_t));
  check_hip(hipMemcpy(tree_ti_, ti.data(), ti.size() * sizeof(int32_t), hipMemcpyHostToDevice),
            "upload tables");
  tree_total_ = g.total;
  tree_depth_ = g.depth;
  if (serves(Precision::FP64)) set_tree_plans<double>(g, mult, multT);
  if (serves(Precision::FP32)) set_tree_plans<float>(g, mult, multT);
  return true;
}

void DeviceMultiEval::release_tree() {
  (void)hipStreamSynchronize(stream_);
  auto drop = [](void** buf, size_t* cap) {
    if (*buf) (void)hipFree(*buf);
    *buf = nullptr;
    *cap = 0;
  };
  drop(&tree_ti_, &tree_ti_cap_);
  for (int ix = 0; ix < 2; ++ix) {
    drop(&tree_x_[ix], &tree_x_cap_[ix]);
    drop(&tree_sperm_[ix], &tree_sperm_cap_[ix]);
    for (TreePlan* p : {&tree_mult_[ix], &tree_multT_[ix]}) {
      drop(&p->recs, &p->recs_cap);
      drop(&p->chunks, &p->chunks_cap);
      drop(&p->groups, &p->groups_cap);
      drop(&p->items, &p->items_cap);
      drop(&p->sums, &p->sums_cap);
    }
  }
}

// ---------------------------------------------------------------- launches

template <typename T>
void DeviceMultiEval::run_tree_mult(const double* d_alpha, double* d_result, hipEvent_t* tev,
                                    const MultScratch* ext) {
  hipStream_t s = stream_;
  const int ix = sizeof(T) == sizeof(double) ? 0 : 1;
  const TreePlan& plan = tree_mult_[ix];
  const TreeLaunch l = basis_ == Basis::ModLinear
                           ? tree_launch<T, true>(static_cast<int>(D_), tree_depth_, tree_wide_[ix])
                           : tree_launch<T, false>(static_cast<int>(D_), tree_depth_, tree_wide_[ix]);
  const int64_t nrows = tree_rows_[ix];
  const unsigned rb = blocks(nrows, kTreeBlock * l.k);
  int G = plan.ngroups, gper = 1;
  // weights in table order first, unless few blocks gather few of them
  const size_t wbytes = (static_cast<size_t>(tree_total_) * sizeof(T) + 255) / 256 * 256;
  bool weights = static_cast<int64_t>(rb) * tree_total_ > (int64_t(1) << 21);
  double* P = nullptr;
  T* W = nullptr;
  if (ext) {
    check_scratch(*ext, sizeof(T));
    if (wbytes > ext->bytes) weights = false;
    const size_t left = ext->bytes - (weights ? wbytes : 0);
    const int64_t rows = static_cast<int64_t>(left / (nrows * sizeof(double)));
    if (rows < G) gper = rows > 1 ? static_cast<int>((G + rows - 1) / rows) : G;
    if (weights) W = static_cast<T*>(ext->base);
    P = reinterpret_cast<double*>(static_cast<unsigned char*>(ext->base) + (weights ? wbytes : 0));
  } else if (weights) {
    ensure(&A_, &A_cap_, wbytes);
    W = static_cast<T*>(A_);
  }
  G = (G + gper - 1) / gper;
  if (G > 1 && !ext) {
    ensure(&part_, &part_cap_, static_cast<size_t>(G) * nrows * sizeof(double));
    P = static_cast<double*>(part_);
  }
  if (weights) {
    clear_launch_error();
    hipLaunchKernelGGL(tree_weights_kernel<T>, dim3(blocks(tree_total_, 256)), dim3(256), 0, s,
                       d_alpha, static_cast<const int32_t*>(tree_ti_), W, tree_total_);
    check_hip(hipGetLastError(), "tree weights");
  }
  TreeMultArgs a{};
  a.X = tree_x_[ix];
  a.ldx = nrows;
  a.D = static_cast<int>(D_);
  a.recs = static_cast<const TreeRec*>(plan.recs);
  a.chunks = static_cast<const TreeChunk*>(plan.chunks);
  a.groups = static_cast<const int*>(plan.groups);
  a.ngroups = plan.ngroups;
  a.gper = gper;
  a.W = W;
  a.alpha = d_alpha;
  a.ti = static_cast<const int32_t*>(tree_ti_);
  a.part = G > 1 ? P : nullptr;
  a.out = d_result;
  a.sperm = static_cast<const int32_t*>(tree_sperm_[ix]);
  a.zero_off = plan.lds;
  if (tev) check_hip(hipEventRecord(tev[0], s), "hipEventRecord");
  l.mult(a, dim3(rb, static_cast<unsigned>(G)), kTreeBlock, static_cast<unsigned>(plan.lds) + 16, s);
  check_hip(hipGetLastError(), "tree mult kernel");
  if (tev) check_hip(hipEventRecord(tev[1], s), "hipEventRecord");
  if (G > 1) {
    clear_launch_error();
    hipLaunchKernelGGL(reduce_rows_kernel, dim3(blocks(nrows, kCols)), dim3(kRows * kCols), 0, s,
                       P, nrows, G, a.sperm, d_result, nrows);
    check_hip(hipGetLastError(), "tree reduce (mult)");
  }
  last_G_ = G;
}

template <typename T>
void DeviceMultiEval::run_tree_multT(const double* d_y, double* d_result, hipEvent_t* tev) {
  hipStream_t s = stream_;
  const int ix = sizeof(T) == sizeof(double) ? 0 : 1;
  const TreePlan& plan = tree_multT_[ix];
  const TreeLaunch l = basis_ == Basis::ModLinear
                           ? tree_launch<T, true>(static_cast<int>(D_), tree_depth_, tree_wide_[ix])
                           : tree_launch<T, false>(static_cast<int>(D_), tree_depth_, tree_wide_[ix]);
  ensure(&Y_, &Y_cap_, Mpad_ * sizeof(T));
  ensure(&part_, &part_cap_, plan.part);
  clear_launch_error();
  hipLaunchKernelGGL(tree_prep_kernel<T>, dim3(blocks(tree_rows_[ix], 256)), dim3(256), 0, s, d_y,
                     static_cast<const int32_t*>(tree_sperm_[ix]), static_cast<T*>(Y_),
                     tree_rows_[ix]);
  check_hip(hipGetLastError(), "tree prep");
  TreeMultTArgs a{};
  a.X = tree_x_[ix];
  a.ldx = tree_rows_[ix];
  a.D = static_cast<int>(D_);
  a.Y = Y_;
  a.recs = static_cast<const TreeRec*>(plan.recs);
  a.chunks = static_cast<const TreeChunk*>(plan.chunks);
  a.items = static_cast<const TreeItem*>(plan.items);
  a.part = static_cast<double*>(part_);
  if (tev) check_hip(hipEventRecord(tev[0], s), "hipEventRecord");
  l.multT(a, static_cast<unsigned>(plan.nitems), static_cast<unsigned>(plan.lds), s);
  check_hip(hipGetLastError(), "tree multTranspose kernel");
  if (tev) check_hip(hipEventRecord(tev[1], s), "hipEventRecord");
  clear_launch_error();
  hipLaunchKernelGGL(tree_sum_kernel, dim3(static_cast<unsigned>(plan.nsums)), dim3(kRows * kCols),
                     0, s, static_cast<const double*>(part_),
                     static_cast<const TreeSum*>(plan.sums),
                     static_cast<const int32_t*>(tree_ti_), d_result);
  check_hip(hipGetLastError(), "tree reduce (multTranspose)");
  last_S_ = plan.segs;
}

template void DeviceMultiEval::run_tree_mult<double>(const double*, double*, hipEvent_t*,
                                                     const MultScratch*);
template void DeviceMultiEval::run_tree_mult<float>(const double*, double*, hipEvent_t*,
                                                    const MultScratch*);
template void DeviceMultiEval::run_tree_multT<double>(const double*, double*, hipEvent_t*);
template void DeviceMultiEval::run_tree_multT<float>(const double*, double*, hipEvent_t*);

}  // namespace sgpp_hip
