// The subspace tree: grids evaluated subspace by subspace, one
// one-dimensional factor per (data point, subspace). Data structures shared by
// the kernels (tree_kernels.hpp), their instantiations and the runtime
// (tree_runtime.hip).
//
// In a subspace W_l (level vector l) the supports of the basis functions tile
// [0,1]^d, so a data point lies in the support of exactly one of them (after
// the reference's SubspaceLinear operator,
// OperationMultipleEvalSubspaceCombined.hpp:92-204). The level vectors form a
// tree: the parent of l is l with its last level above 1 set to 1, so a
// subspace's basis value is its parent's times ONE factor, and its table
// position is its parent's extended by one cell number. The subspaces are kept
// in depth-first order, a parent's children by dimension, then level.
//
// A program is the tree's nodes as 16-byte records in that order; a wave walks
// it with one or more data points per lane, the parents' products and table
// positions in registers, one set per depth.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <vector>

#include "meval_device.hpp"
#include "subspace_device.hpp"

namespace sgpp_hip {

// Levels above 1 of one level vector at most (the register sets of a walk);
// deeper grids are left to the other kernels.
constexpr int kTreeMaxDepth = 12;
// of the usual walks
constexpr int tree_few_dims(size_t D) { return D <= 4 ? 4 : 6; }

// threads of a mult block (four waves share one chunk's tables)
constexpr int kTreeBlock = 256;

// multTranspose joins the values of 2^kTreeJoin lanes
constexpr int kTreeJoin = 1;

// ctl of a record
// bits 0 to 4: 33 - level
constexpr int kTreeDimShift = 8;            // 6 bits: the dimension
constexpr uint32_t kTreeRun = 1u << 16;     // first of its (parent, dimension): fetch its values
constexpr uint32_t kTreeTable = 1u << 17;   // the subspace has grid points (absent parents are walked without)
constexpr uint32_t kTreePush = 1u << 18;    // children follow
constexpr uint32_t kTreeLast = 1u << 19;    // last of its parent's children
constexpr uint32_t kTreeFlush = 1u << 20;   // add the FP32 sums to the FP64 ones
constexpr uint32_t kTreePart = 1u << 21;    // (without kTreeTable) part of a table: see TreeChunk
constexpr int kTreePassShift = 24;          // 4 bits: the dimensions before the run's to pass first

// Linear grids of up to this many dimensions are walked with the product of the
// factors of the dimensions passed, those of more with the product of all, of which
// a run takes its own dimension's level-1 factor out: three roundings per refined
// dimension and one, where the product of D factors has D - 1. RMS error of the basis
// values in 2^-53 (FP32: 2^-24, alike), culled kernels, dimensions passed, factor taken out:
//   d=2  level 8     0.49  0.42  0.98     d=11 20,000 points  1.59  1.31  1.47
//   d=5  level 7     0.98  0.84  1.30     d=20 level 4        3.26  1.80  1.64
//   d=9  20,000 points 1.42 1.22 1.56     d=30 level 3        3.68  2.17  0.92
// (Taken out of a product of all below 2^-126, FP32 values lose digits: basis values
// below 2^-96; a coordinate below 2^-127 counts as 0.)
constexpr int kTreePassDims = 10;

struct alignas(16) TreeRec {
  uint32_t off;    // byte offset of the subspace's table in the chunk's LDS image
  uint32_t ctl;
  uint32_t scale;  // 2^(level - 1) / 2^32: the float's bits, or the double's upper word
  uint32_t pad;
};
static_assert(sizeof(TreeRec) == 16, "one record is 16 bytes");

// A run of consecutive subspaces whose tables fit the LDS image: records
// [rec0, rec0 + nrec), table entries [off0, off0 + n). root: the chunk begins
// with the subspace of level 1 in every dimension (one entry, the first). Of a
// subspace whose table exceeds the image a chunk holds positions [part0, part0 + n).
struct alignas(16) TreeChunk {
  int rec0, nrec;
  int n, part0;
  long long off0;
  int root, pad;
};
static_assert(sizeof(TreeChunk) == 32, "one chunk is 32 bytes");

// A multTranspose block: batches [b0, b1) of 64 * K rows for one chunk, whose
// sums go to part[off, off + n).
struct alignas(16) TreeItem {
  int chunk, b0, b1, pad;
  long long off, pad2;
};
static_assert(sizeof(TreeItem) == 32, "one item is 32 bytes");

// The partial sums of up to 64 table entries of a chunk: rows of stride ld, the
// first at off; entries [e0, e0 + n) of the tables.
struct alignas(16) TreeSum {
  int n, rows;
  long long off, ld, e0;
};
static_assert(sizeof(TreeSum) == 32, "one sum is 32 bytes");

// A grid's subspaces in walking order, and their tables.
struct TreeGrid {
  struct Node {
    int depth;             // levels above 1
    int64_t off;           // table offset
    int bits;              // table entries: 2^bits
  };
  size_t D = 0;
  std::vector<uint8_t> level;  // [nodes][D]
  std::vector<Node> node;
  std::vector<uint32_t> order; // the grid points by node
  std::vector<uint32_t> first; // per node its first in order, and their number
  int64_t total = 0;           // table entries
  int depth = 0;               // of the deepest node
};
// Sorts the points of a no-boundary grid by subspace. False for grids that the walks
// do not cover: more than kTreeMaxDepth levels above 1 in a level vector, tables
// beyond subspace_table_limit(N) or 2^30 cells in one subspace.
bool build_tree_grid(size_t D, size_t N, const uint32_t* level, TreeGrid& g);
// The grid point of every table entry, or -1; false if a grid point occurs twice
// (a table holds it once).
bool tree_tables(const TreeGrid& g, const uint32_t* level, const uint32_t* index,
                 std::vector<int32_t>& ti);

// Nodes to walk per data point, those of tables in parts counted per part (and
// their ancestors).
int64_t tree_walks(const TreeGrid& g, bool multT);

// Programs of a grid: groups of chunks of at most cap table entries and
// max_nodes nodes; the groups have about equal numbers of nodes.
struct TreeProgram {
  std::vector<TreeRec> recs;
  std::vector<TreeChunk> chunks;
  std::vector<int> groups;
  int max_entries = 0;
};
TreeProgram build_tree_program(const TreeGrid& g, int ngroups, int64_t cap, int64_t max_nodes,
                               int entry_bytes, bool fp32);

struct TreeMultArgs {
  const void* X;  // [rows of ldx]: tree_points_kernel
  int64_t ldx;
  int D;
  const TreeRec* recs;
  const TreeChunk* chunks;
  const int* groups;  // chunk group g: chunks [groups[g], groups[g + 1])
  int ngroups, gper;  // groups, and groups per block (blockIdx.y)
  const void* W;      // weights in table order and compute type, or null:
  const double* alpha;  // gathered from here through ti
  const int32_t* ti;
  double* part;  // [gridDim.y][ldx], or null: results to out[sperm[row]]
  double* out;
  const int32_t* sperm;  // the caller's row, -1 for padding
  int zero_off;  // byte offset of an LDS zero (rows outside a part)
};

struct TreeMultTArgs {
  const void* X;
  int64_t ldx;
  int D;
  const void* Y;  // [ldx] in X's order and type, 0 in padding rows
  const TreeRec* recs;
  const TreeChunk* chunks;
  const TreeItem* items;  // one per block
  double* part;
};

// Launchers of one compute type and basis. wide: several data points per
// lane; D: dimensions, depth: of the grid's tree. rows(): data points per
// wave.
struct TreeLaunch {
  int k = 1;
  void (*mult)(const TreeMultArgs&, dim3 grid, unsigned block, unsigned lds, hipStream_t s) = nullptr;
  void (*multT)(const TreeMultTArgs&, unsigned items, unsigned lds, hipStream_t s) = nullptr;
};
template <typename T, bool kMod>
TreeLaunch tree_launch(int D, int depth, bool wide);
extern template TreeLaunch tree_launch<float, false>(int, int, bool);
extern template TreeLaunch tree_launch<float, true>(int, int, bool);
extern template TreeLaunch tree_launch<double, false>(int, int, bool);
extern template TreeLaunch tree_launch<double, true>(int, int, bool);

}  // namespace sgpp_hip
