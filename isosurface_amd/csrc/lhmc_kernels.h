// Launch interface of the linear-hashed octree marching-cubes kernels.
//
// The octree is built breadth first; its nodes live in one array, depth by
// depth, families of eight together (in Morton order), the families of a depth
// in no order.  Primal vertices are listed in ascending key order: for shallow
// trees by marking a bit lattice at depth max_depth + 1 indexed by Morton code
// and scanning it, for deeper ones by sorting the leaves' (vertex, level) pairs.
// Dual cubes are then processed in that order with an open-addressing table over
// their edges.
//
// Node, vertex and cube counts pass from launch to launch in device memory
// (LhmcTree::ctl).  A launch whose results outgrow a buffer leaves out the
// writes that do not fit, and the ones after it do nothing; the host sees the
// counts, grows the buffer and starts over.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "scan.h"
#include "sdf_program.h"
#include "sparse_kernels.h"

namespace iso {

// Nodes reach depth max_depth + 1, whose keys need 3 (max_depth + 1) + 1
// bits: 20 is the deepest whose keys fit 64 bits (the reference's MAX_LEVEL
// is 21).
constexpr int kLhmcMaxDepth = 20;
constexpr int kLhmcMaxLevels = kLhmcMaxDepth + 2;  // depths 0 .. max(2, max_depth) + 1
// Trees whose primal bit lattice (8^(max(2, max_depth) + 1) bits) would
// exceed this many levels take the sorted primal path.
constexpr int kLhmcDenseDepth = 9;

// Status bits written by the LHMC kernels.
enum : unsigned long long {
  kLhmcErrScan = 2ull,        // a look-back gave up (scan::State::err)
  kLhmcErrTable = 8ull,       // edge table full
};

// Words of LhmcTree::ctl.
enum : int {
  kLhmcCount = 0,    // nodes of each depth
  kLhmcPrimal = 24,  // [ticket, primal vertices]
  kLhmcCubes = 26,   // [ticket, listed cubes << 32 | triangles]
  kLhmcOwn = 28,     // [ticket, vertices]
  kLhmcErr = 30,     // status bits
  kLhmcCtlWords = 32,
};
static_assert(kLhmcMaxLevels + 1 <= kLhmcPrimal, "a word for every depth");

constexpr uint32_t kLhmcLeaf = 0xffffffffu;

struct LhmcTree {
  const DevOp* ops;
  int n_ops;
  int max_depth;
  int d1;                   // the deepest a node can be
  uint64_t cap;             // nodes that keys, values and child hold
  uint64_t* keys;           // Morton keys (0: no node)
  float* values;            // SDF at each node's (quirky) centre
  uint32_t* child;          // first of the eight children, kLhmcLeaf if not refined
  const uint64_t* split;    // lhmc_level_splits
  uint32_t* bits;           // primal lattice of depth d1, a bit a vertex; null: sorted path
  unsigned long long* ctl;  // kLhmcCtlWords
};

struct LhmcEdgeTable {
  unsigned long long* keys;  // (node a << 32) | node b, a < b; ~0 = empty
  uint32_t* owner;           // least 16 * cube + listing order of those that use the edge
  uint32_t* id;              // vertex id
  uint64_t mask;             // slots in use - 1: lhmc_table_size() - 1
};

// Slots that the edges of some cubes need, by their LhmcTree::ctl word: a power
// of two, at least twice the edges that their triangles can have (at most 12
// edges a cube: fewer than 2^32 in all).
__host__ __device__ inline uint64_t lhmc_table_size(uint64_t cubes_word) {
  const uint64_t want = 6 * (cubes_word & 0xffffffffull);
  if (want <= 1024) return 1024;
  const uint64_t size = 1ull << (64 - __builtin_clzll(want - 1));
  return size < (1ull << 32) ? size : 1ull << 32;
}

struct LhmcCubes {
  uint64_t* primal;            // Morton key (MAX_LEVEL) of each primal vertex, ascending
  uint8_t* primal_level;       // its deepest touching leaf level (sorted path)
  uint64_t primal_capacity;    // vertices that these hold
  uint64_t capacity;           // cubes that the arrays below hold (those with triangles)
  uint32_t* corner;            // 8 node indices per cube
  uint32_t* edge_slot;         // 12 table slots per cube
  uint32_t* tri_first;         // triangles of the cubes before it
  uint8_t* cube_case;          // cube index
  uint64_t table_capacity;     // slots of the edge table
  unsigned long long* slot;    // scan slots: primal_capacity / 1024 + 1
  unsigned long long* own_slot;  // and capacity / 256 + 1
};

// Morton::level() (morton.rs:53-59) takes floor(ln(key) * 0.48089834696)
// in f64; the truncated constant puts the first split[d] keys of depth d,
// [8^d, 8^d + split[d]), one level low.  lhmc_level_splits() finds split[d]
// on the host with the same libm log the reference uses (1 for d <= 10, then
// 2, 11, 93, ... up to 2502362113 at d = 21); the kernels read the table.
void lhmc_level_splits(uint64_t split[kLhmcMaxLevels]);

// Clears ctl, n_slots scan slots, and the bit lattice.
hipError_t launch_lhmc_clear(const LhmcTree& T, unsigned long long* slot, uint64_t n_slots,
                             hipStream_t s);
// Nodes of every depth, their values and children; on the bit lattice the
// leaves' primal vertices.
hipError_t launch_lhmc_levels(const LhmcTree& T, const ProgramKind& kind, hipStream_t s);
// Lists the marked vertices in ascending order.  `slot`: lhmc_primal_slots(d1)
// cleared scan slots.
uint64_t lhmc_primal_slots(int d1);
hipError_t launch_lhmc_primal(const LhmcTree& T, const LhmcCubes& C, unsigned long long* slot,
                              hipStream_t s);
// The same list without a lattice: every node writes 8 (vertex, level) pairs
// (key 0 for none) into pair_keys / pair_levels (8 * n_nodes each), a radix
// sort orders them into sorted_keys / sorted_levels, and the last pair of each
// run of equal keys (with the run's deepest level) is listed.  `temp` holds
// lhmc_sort_temp_bytes(8 * n_nodes) bytes, `slot` a slot for every 2048 pairs.
size_t lhmc_sort_temp_bytes(uint64_t n_pairs);
hipError_t launch_lhmc_primal_sorted(const LhmcTree& T, int64_t n_nodes, uint64_t* pair_keys,
                                     uint8_t* pair_levels, uint64_t* sorted_keys,
                                     uint8_t* sorted_levels, void* temp, size_t temp_bytes,
                                     const LhmcCubes& C, unsigned long long* slot, hipStream_t s);
// Cube corners and cases, and the list of the cubes with triangles
// (`launch_lhmc_cubes_reset` first where the clear did not cover its slots).
hipError_t launch_lhmc_cubes_reset(const LhmcTree& T, const LhmcCubes& C, hipStream_t s);
hipError_t launch_lhmc_cubes(const LhmcTree& T, const LhmcCubes& C, hipStream_t s);
// Edge ownership (first cube), vertex ids and positions.  May be run again
// after launch_lhmc_cubes, with a larger table or more room for vertices.
hipError_t launch_lhmc_own(const LhmcTree& N, const LhmcCubes& C, const LhmcEdgeTable& T,
                           float* vertices, uint64_t vcap, hipStream_t s);
// Index triples.
hipError_t launch_lhmc_emit(const LhmcTree& N, const LhmcCubes& C, const LhmcEdgeTable& T,
                            uint32_t* indices, uint64_t icap, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s);

}  // namespace iso
