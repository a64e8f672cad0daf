// Linear-hashed octree marching cubes for gfx950 (MI355X).
//
// LinearHashedMarchingCubes::extract (linear_hashed_marching_cubes.rs:62-84)
// over ImplicitOctree::traverse (traversal/implicit_octree.rs:39-99):
//   1. level    per depth: sample each node at its Morton centre, decide
//               refinement (implicit_octree.rs:47-59), scan the decisions
//               and write the refined nodes' children in key order.  Depths 0
//               to 3 are one workgroup's work, the next ones a launch each,
//               every launch taking its extent from the one before in device
//               memory.  Leaves mark their primal vertices (morton.rs:120-138)
//               in a bit lattice with the deepest possible spacing;
//   2. primal   a scan over the lattice's words lists the vertices in
//               ascending Morton order;
//   3. cubes    per primal vertex the eight dual corners (morton.rs:142-146),
//               each the deepest existing node on its parent chain, which
//               eight descents from the root by child index find together;
//               cube index; the cubes with triangles are listed, in order;
//   4. own      each dual-cube edge (MortonKey, index_cache.rs:63-73) is owned
//               by the first cube, in order, whose triangles use it (a hash
//               table, whose slots the cubes keep); owned edges are counted,
//               scanned into first ids, and their crossings written;
//   5. emit     every listed cube writes its index triples.
// All steps are queued together, and one round trip tells the host the sizes.
// Latency bounds this path (a few thousand to a few hundred thousand nodes):
// depth 7 of the union of 32 boxes took 917 us in 60 launches and copies with 13
// round trips, of which 131 us scanned 16.7 M lattice words and 133 us searched
// sorted keys by bisection; now 249 us in fourteen launches.
// The output is the reference's for the primal-vertex order "ascending
// Morton key" (the reference's own order is a std HashMap's, random per
// process).  Morton::level() keeps the reference's quirk: the truncated
// constant 0.48089834696 (morton.rs:35, 54-59) puts the first keys of each
// depth one level low (exactly the power of 8 below 8^11, then more: a
// table of split points found with the host's libm log).  Deep trees
// (beyond kLhmcDenseDepth) list their primal vertices by a radix sort of
// the leaves' (vertex, level) pairs instead of a bit lattice.  A node is refined while its level is
// below M = max(2, max_depth); the origin-corner node of depth M has level
// M - 1, so nodes reach depth M + 1, the "dense depth" of the primal lattice.
#include <hip/hip_runtime.h>

#include <cmath>
#include <rocprim/device/device_radix_sort.hpp>

#include "lhmc_kernels.h"
#include "mc_tables.h"
#include "sparse_eval.h"

namespace iso {

namespace {

// morton.rs:17-32
constexpr uint64_t kMask2 = 0x7FC0000FF80001FFull;
constexpr uint64_t kMask1 = 0x01C0E070381C0E07ull;
constexpr uint64_t kMask0 = 0x9249249249249249ull;
constexpr uint64_t kTz = 0x4924924924924924ull;
constexpr uint64_t kTy = 0x2492492492492492ull;
constexpr uint64_t kTx = 0x9249249249249249ull;
constexpr uint64_t kT1 = 0xB6DB6DB6DB6DB6DBull;
constexpr uint64_t kT2 = 0xDB6DB6DB6DB6DB6Dull;
constexpr uint64_t kT3 = 0x6DB6DB6DB6DB6DB6ull;
constexpr int kMaxLevel = 21;
constexpr float kSqrtOf3 = 1.73205080757f;  // distance.rs:18
constexpr unsigned long long kEmpty = ~0ull;
// Bits 8 p of a lattice word whose vertex p is not on the word's low face
// along an axis.
constexpr uint64_t word_bits(uint64_t axis) {
  uint64_t m = 0;
  for (uint64_t p = 0; p < 8; ++p)
    if (p & axis) m |= 1ull << (8 * p);
  return m;
}
constexpr uint64_t kAlongX = word_bits(kTx & 7), kAlongY = word_bits(kTy & 7),
                   kAlongZ = word_bits(kTz & 7);

__constant__ tables::McTables c_lt = tables::kTables;

__device__ __forceinline__ int depth_of(uint64_t k) { return (63 - __clzll(k)) / 3; }

// Morton::level() (morton.rs:53-59): the depth, one less for the first
// split[d] keys of depth d.
__device__ __forceinline__ int level_of(const uint64_t* split, uint64_t k) {
  if (k == 0) return 0;
  const int d = depth_of(k);
  return (d >= 1 && k - (1ull << (3 * d)) < split[d]) ? d - 1 : d;
}

__device__ __forceinline__ float size_at(int level) {  // morton.rs:73-75
  return 1.0f / static_cast<float>(2ull << level);
}

struct F3 {
  float x, y, z;
};

__device__ __forceinline__ F3 center_of(uint64_t k, int lv) {  // morton.rs:78-116
  uint64_t bz = (k >> 2) & kMask0;
  uint64_t by = (k >> 1) & kMask0;
  uint64_t bx = k & kMask0;
  if (lv > 1) {
    bz = (bz | (bz >> 2) | (bz >> 4)) & kMask1;
    by = (by | (by >> 2) | (by >> 4)) & kMask1;
    bx = (bx | (bx >> 2) | (bx >> 4)) & kMask1;
    if (lv > 3) {
      bz = (bz | (bz >> 6) | (bz >> 12)) & kMask2;
      by = (by | (by >> 6) | (by >> 12)) & kMask2;
      bx = (bx | (bx >> 6) | (bx >> 12)) & kMask2;
      if (lv > 9) {
        bz = bz | (bz >> 18) | (bz >> 36);
        by = by | (by >> 18) | (by >> 36);
        bx = bx | (bx >> 18) | (bx >> 36);
      }
    }
  }
  const uint64_t length_mask = (1ull << lv) - 1;
  bz &= length_mask;
  by &= length_mask;
  bx &= length_mask;
  const float s = size_at(lv);
  const float s2 = s * 2.0f;
  return {static_cast<float>(bx) * s2 + s, static_cast<float>(by) * s2 + s,
          static_cast<float>(bz) * s2 + s};
}

__device__ __forceinline__ uint64_t m_add(uint64_t a, uint64_t b) {  // morton.rs:153-163
  return (((a | kT1) + (b & kTz)) & kTz) | (((a | kT2) + (b & kTy)) & kTy) |
         (((a | kT3) + (b & kTx)) & kTx);
}

__device__ __forceinline__ uint64_t m_sub(uint64_t a, uint64_t b) {  // morton.rs:165-175
  return (((a & kTz) - (b & kTz)) & kTz) | (((a & kTy) - (b & kTy)) & kTy) |
         (((a & kTx) - (b & kTx)) & kTx);
}

__device__ __forceinline__ uint64_t primal_vertex(uint64_t key, int lv, unsigned which) {
  const uint64_t k = 1ull << (3 * lv);  // morton.rs:120-138
  const uint64_t k_plus_one = k << 1;
  const uint64_t vk = m_add(key, which);
  const uint64_t dk = m_sub(vk, k);
  if (vk >= k_plus_one || (dk & kTx) == 0 || (dk & kTy) == 0 || (dk & kTz) == 0) return 0;
  return vk << (3 * (kMaxLevel - lv));
}

__device__ __forceinline__ uint64_t dual_vertex(uint64_t key, int lv, unsigned which) {
  return m_sub(key >> (3 * (kMaxLevel - lv)), which);  // morton.rs:142-146
}

__device__ __forceinline__ uint64_t hash_edge(unsigned long long k) {
  k ^= k >> 33;
  k *= 0xff51afd7ed558ccdull;
  k ^= k >> 33;
  k *= 0xc4ceb9fe1a85ec53ull;
  k ^= k >> 33;
  return k;
}

// Slot of edge key `k`, inserting it if absent; ~0 if the table is full.
__device__ __forceinline__ uint64_t table_insert(const LhmcEdgeTable& T, unsigned long long k) {
  uint64_t h = hash_edge(k) & T.mask;
  for (uint64_t probe = 0; probe <= T.mask; ++probe) {
    // (most edges are in already: a key read late only costs the exchange)
    if (T.keys[h] == k) return h;
    const unsigned long long cur = atomicCAS(&T.keys[h], kEmpty, k);
    if (cur == kEmpty || cur == k) return h;
    h = (h + 1) & T.mask;
  }
  return ~0ull;
}

__device__ __forceinline__ unsigned long long edge_key(const uint32_t* corner, int e) {
  uint32_t a = corner[tables::kEdgeCorners[e][0]], b = corner[tables::kEdgeCorners[e][1]];
  if (a > b) {
    const uint32_t t = a;
    a = b;
    b = t;
  }
  return (static_cast<unsigned long long>(a) << 32) | b;
}

// ---- 1. octree depths -------------------------------------------------------
// The SDF at a node's centre; every lane of the wavefront takes part.  kKind:
// 0 any program, 1 bounded without a stack, 2 bounded with one.  Nodes that
// follow each other in Morton order lie close together, and few operations of
// a union can change a value in their box.  (Every launch here is one such
// evaluation's latency: 32 boxes one after the other, each read from memory,
// took 13 us.)  `head`: node_ops, read early.
template <int kKind>
__device__ __forceinline__ DevOp node_ops(const LhmcTree& T) {
  return kKind ? lane_ops(as_constant(T.ops), 0, T.n_ops) : DevOp{};
}
template <int kKind>
__device__ __forceinline__ float node_value(const LhmcTree& T, const DevOp& head, const F3& c) {
  if constexpr (kKind == 0) {
    return sdf_eval(T.ops, T.n_ops, c.x, c.y, c.z);
  } else {
    const float p[1][3] = {{c.x, c.y, c.z}};
    float v[1];
    sdf_eval_near<1, kKind == 2>(as_constant(T.ops), T.n_ops, head, p, v);
    return v[0];
  }
}

// Signed::within_extent (distance.rs:60-62)
__device__ __forceinline__ bool refined(int level, int max_depth, float v) {
  return level < 2 || (level < max_depth && __builtin_fabsf(v) < size_at(level) * kSqrtOf3);
}

// Marks the primal vertices of leaf `key` of depth and level d.  `family`:
// which of its eight siblings are such leaves, by child index; a vertex that
// several of them share is marked by the first (27 marks a family, not 64).
__device__ __forceinline__ void mark_leaf(const LhmcTree& T, uint64_t key, int d, uint32_t family) {
  const uint64_t lmask = (1ull << (3 * T.d1)) - 1;
  const uint32_t c = static_cast<uint32_t>(key & 7);
#pragma unroll
  for (uint32_t w = 0; w < 8; ++w) {
    uint32_t share = family;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t high = a == 0 ? 0xAAu : a == 1 ? 0xCCu : 0xF0u;  // siblings with bit a
      if (((c ^ w) >> a & 1) == 0) share &= (c >> a & 1) ? high : ~high;
    }
    if (static_cast<uint32_t>(__builtin_ctz(share)) != c) continue;
    const uint64_t v = primal_vertex(key, d, w);
    if (v == 0) continue;
    const uint64_t at = (v >> (3 * (kMaxLevel - T.d1))) & lmask;
    const uint32_t bit = 1u << (at & 31);
    atomicOr(&T.bits[at >> 5], bit);
  }
}

// The same for all leaves of a family at depth d1 - 1, most of a tree's, whose
// low vertices make up one 64-bit word of the lattice: lane c of the family
// marks the vertices in the word c of the eight around it.  `origin`: the
// family's first key.  (Some of the words do not exist, past the high faces of
// the domain, and some vertices do not count, on its low faces.)
__device__ __forceinline__ void mark_family(const LhmcTree& T, uint64_t origin, uint32_t family,
                                            uint32_t c) {
  const int d = T.d1 - 1;
  uint64_t bits = 0;
#pragma unroll
  for (uint32_t p = 0; p < 8; ++p) {
    if (p & c) continue;  // the vertex's low bits: 0 along the axes where it is in the next word
    uint32_t share = family;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const uint32_t high = a == 0 ? 0xAAu : a == 1 ? 0xCCu : 0xF0u;
      if (c >> a & 1) share &= high;
      else if (!(p >> a & 1)) share &= ~high;
    }
    if (share) bits |= 1ull << (8 * p);
  }
  if (!bits) return;
  // morton.rs:120-138 for the word's vertices together
  const uint64_t k = 1ull << (3 * d);
  const uint64_t word = m_add(m_add(origin, c), c);  // + 2 along c's axes
  if (word >= k << 1) return;
  const uint64_t dk = m_sub(word, k);
  if ((dk & kTx) == 0) bits &= kAlongX;
  if ((dk & kTy) == 0) bits &= kAlongY;
  if ((dk & kTz) == 0) bits &= kAlongZ;
  if (!bits) return;
  atomicOr(reinterpret_cast<unsigned long long*>(T.bits) + ((word & (k - 1)) >> 3), bits);
}

// Room for the children of a wavefront's `refining` nodes, in whatever order
// the wavefronts come: nothing that follows depends on the order of the nodes.
// Returns the first child of this lane's node.
__device__ __forceinline__ uint64_t child_room(const LhmcTree& T, int d, uint64_t end, bool ref) {
  const uint64_t refining = __ballot(ref);
  if (!refining) return 0;
  unsigned long long first = 0;
  if (__lane_id() == 0)
    first = atomicAdd(&T.ctl[kLhmcCount + d + 1], 8ull * __popcll(refining));
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(first));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(first >> 32));
  return end + (static_cast<uint64_t>(hi) << 32 | lo) +
         8 * __popcll(refining & ((1ull << __lane_id()) - 1));
}

__device__ __forceinline__ void write_children(const LhmcTree& T, uint64_t at, uint64_t key) {
  if (at + 8 > T.cap) return;
#pragma unroll
  for (unsigned c = 0; c < 8; ++c) T.keys[at + c] = (key << 3) | c;
}

// Depths 0 to 3 as 10 workgroups of one wavefront: the first two depths always
// refine (implicit_octree.rs:47-59), so all 585 candidates have their places.
// The wavefronts of depth 3 evaluate their parents too; a node whose parent
// does not refine has key 0.
template <int kKind>
__global__ __launch_bounds__(64) void k_top(LhmcTree T) {
  const DevOp head = node_ops<kKind>(T);
  const int lane = __lane_id();
  const bool deep = blockIdx.x >= 2;  // (one depth a wavefront, so families are whole)
  const int rel0 = deep ? 64 * (static_cast<int>(blockIdx.x) - 2) + lane : lane;
  if (!deep && blockIdx.x == 0) {  // depths 0 and 1
    const int t = lane < 9 ? lane : 8, d = t ? 1 : 0;
    const uint64_t key = d ? 8 + (t - 1) : 1;
    const float v = node_value<kKind>(T, head, center_of(key, level_of(T.split, key)));
    if (lane < 9) {
      T.keys[t] = key;
      T.values[t] = v;
      T.child[t] = d ? 9 + 8 * (t - 1) : 1;
    }
    if (lane < 4)
      T.ctl[kLhmcCount + lane] = lane == 0 ? 1 : lane == 1 ? 8 : lane == 2 ? 64 : 512;
    return;
  }
  const int d = deep ? 3 : 2;
  const uint64_t key = (1ull << (3 * d)) | static_cast<uint64_t>(rel0);
  const int lv = level_of(T.split, key);
  bool exists = true;
  if (deep) {
    const int plv = level_of(T.split, key >> 3);
    exists = refined(plv, T.max_depth,
                     node_value<kKind>(T, head, center_of(key >> 3, plv)));
  }
  const float v = node_value<kKind>(T, head, center_of(key, lv));
  const bool ref = exists && refined(lv, T.max_depth, v);
  const int at = (deep ? 73 : 9) + rel0;
  uint32_t child = kLhmcLeaf;
  if (deep) {
    const uint64_t room = child_room(T, 3, 585, ref);
    if (ref) {
      child = static_cast<uint32_t>(room);
      write_children(T, room, key);
    }
  } else if (ref) {
    child = 73 + 8 * rel0;
  }
  T.keys[at] = exists ? key : 0;
  T.values[at] = v;
  T.child[at] = child;
  const bool marks = exists && !ref && lv == d;
  const uint32_t family = static_cast<uint32_t>(__ballot(marks) >> (lane & 56)) & 0xFFu;
  if (marks && T.bits) mark_leaf(T, key, d, family);
}

// One depth from 4 on, whose extent the depths before it have counted.  Small
// depths take a wavefront a workgroup: their time is one evaluation, and a
// compute unit to itself makes that shortest.
template <int kKind, int W>
__global__ __launch_bounds__(64 * W) void k_level(LhmcTree T, int d) {
  const DevOp head = node_ops<kKind>(T);
  uint64_t first = 0;
  for (int i = 0; i < d; ++i) first += T.ctl[kLhmcCount + i];
  const uint64_t n = T.ctl[kLhmcCount + d], end = first + n;
  if (end > T.cap) return;  // this depth, or one above, did not fit
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * 64 * W;
  for (uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * 64 * W + (threadIdx.x & ~63u); i0 < n;
       i0 += stride) {
    const uint64_t i = i0 + __lane_id();
    const bool in = i < n;
    const uint64_t node = first + (in ? i : n - 1);
    const uint64_t key = T.keys[node];
    const int lv = key - (1ull << (3 * d)) < T.split[d] ? d - 1 : d;
    const float v = node_value<kKind>(T, head, center_of(key, lv));
    const bool ref = in && refined(lv, T.max_depth, v);
    const uint64_t room = child_room(T, d, end, ref);
    if (in) {
      T.values[node] = v;
      T.child[node] = ref ? static_cast<uint32_t>(room) : kLhmcLeaf;
      if (ref && d < T.d1) write_children(T, room, key);
    }
    if (T.bits) {  // (depths above 0 come in whole families of eight, aligned)
      const bool marks = in && !ref && lv == d;
      const uint32_t family =
          static_cast<uint32_t>(__ballot(marks) >> (__lane_id() & 56)) & 0xFFu;
      if (d == T.d1 - 1) {
        if (in && family) mark_family(T, key & ~7ull, family, static_cast<uint32_t>(key & 7));
      } else if (marks) {
        mark_leaf(T, key, d, family);
      }
    }
  }
}

// Workgroups of the passes below: sixteen wavefronts, so that a pass over a
// hundred thousand items takes a hundred tickets.  (Tickets are atomics on one
// word, 10 to 20 ns each, whatever else the chip does; with 256 threads they
// were half of such a pass.)
constexpr int kTile = 1024;
constexpr int kTileWaves = kTile / 64;

struct TileShared {
  uint32_t tile;
  unsigned long long wave[kTileWaves];
  unsigned long long prefix;
};

// Tiles in ticket order, until none is left.  A grid that has a workgroup for
// every tile takes no more tickets than tiles.
__device__ __forceinline__ bool next_tile(unsigned long long* ticket, uint64_t n_tiles,
                                          TileShared& S, bool first, uint64_t* tile) {
  if (n_tiles <= gridDim.x && (!first || blockIdx.x >= n_tiles)) return false;
  if (threadIdx.x == 0) S.tile = atomicAdd(reinterpret_cast<unsigned int*>(ticket), 1u);
  __syncthreads();
  *tile = S.tile;
  return *tile < n_tiles;
}

// Exclusive prefix over the workgroup's threads and the workgroups before it;
// *upto receives the prefix after this workgroup.
__device__ __forceinline__ unsigned long long scan_tile(unsigned long long v, uint64_t tile,
                                                        unsigned long long* slot,
                                                        unsigned long long* err, TileShared& S,
                                                        unsigned long long* upto) {
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  unsigned long long inc = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const unsigned long long o = __shfl_up(inc, d, 64);
    if (lane >= d) inc += o;
  }
  if (lane == 63) S.wave[wv] = inc;
  __syncthreads();
  unsigned long long off = inc - v, total = 0ull;
#pragma unroll
  for (int i = 0; i < kTileWaves; ++i) {
    if (i < wv) off += S.wave[i];
    total += S.wave[i];
  }
  if (wv == 0) {
    const unsigned long long prefix = scan::look_back(tile, total, slot, err);
    if (lane == 0) S.prefix = prefix;
  }
  __syncthreads();
  *upto = S.prefix + total;
  return S.prefix + off;
}

// ---- 2. primal vertices -----------------------------------------------------
__device__ __forceinline__ uint64_t lane_word(uint64_t x, int from) {
  const uint32_t lo = __builtin_amdgcn_readlane(static_cast<uint32_t>(x), from);
  const uint32_t hi = __builtin_amdgcn_readlane(static_cast<uint32_t>(x >> 32), from);
  return static_cast<uint64_t>(hi) << 32 | lo;
}

// A word a lane; then the wavefront writes its words' vertices, a word at a
// time, a lane a bit.
__global__ __launch_bounds__(kTile) void k_list(LhmcTree T, LhmcCubes C, uint64_t n_words,
                                                unsigned long long* slot) {
  __shared__ TileShared S;
  const uint64_t* words = reinterpret_cast<const uint64_t*>(T.bits);
  const uint64_t n_tiles = (n_words + kTile - 1) / kTile;
  const int lane = __lane_id();
  uint64_t tile;
  for (bool more = true; next_tile(&T.ctl[kLhmcPrimal], n_tiles, S, more, &tile); more = false) {
    const uint64_t i = tile * kTile + threadIdx.x;
    const uint64_t word = i < n_words ? words[i] : 0ull;
    unsigned long long upto;
    const unsigned long long ex =
        scan_tile(__popcll(word), tile, slot, &T.ctl[kLhmcErr], S, &upto);
    if (tile + 1 == n_tiles && threadIdx.x == 0) T.ctl[kLhmcPrimal + 1] = upto;
    for (uint64_t todo = __ballot(word != 0); todo; todo &= todo - 1) {
      const int from = static_cast<int>(__builtin_ctzll(todo));
      const uint64_t w = lane_word(word, from);
      const uint64_t at = lane_word(ex, from) + __popcll(w & ((1ull << lane) - 1));
      // the lattice index back to the vertex's Morton key at MAX_LEVEL
      if ((w >> lane & 1) && at < C.primal_capacity)
        C.primal[at] = ((64 * (i - lane + from) + lane) | (1ull << (3 * T.d1)))
                       << (3 * (kMaxLevel - T.d1));
    }
  }
}

// Sorted path: every node's eight primal vertices as (key, level) pairs;
// a node that is not a leaf, or a vertex outside the domain, writes key 0
// (every primal key has bit 63 set, so 0 sorts first and marks none).
__global__ __launch_bounds__(256) void k_primal_pairs(LhmcTree T, int64_t n_nodes,
                                                      uint64_t* __restrict__ keys,
                                                      uint8_t* __restrict__ levels) {
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n_nodes;
       i += stride) {
    const uint64_t key = T.keys[i];
    const bool leaf = key != 0 && T.child[i] == kLhmcLeaf;
    const int lv = level_of(T.split, key);
    for (unsigned w = 0; w < 8; ++w) {
      const uint64_t v = leaf ? primal_vertex(key, lv, w) : 0ull;
      keys[8 * i + w] = v;
      levels[8 * i + w] = static_cast<uint8_t>(lv);
    }
  }
}

// The last pair of each run of equal nonzero keys (a vertex is shared by at
// most eight leaves), listed with the run's deepest level.
struct RunLoad {
  const uint64_t* keys;
  uint64_t n;
  __device__ unsigned long long operator()(uint64_t i) const {
    const uint64_t k = keys[i];
    return (k != 0 && (i + 1 == n || keys[i + 1] != k)) ? 1ull : 0ull;
  }
};

struct RunSink {
  const uint64_t* keys;
  const uint8_t* levels;
  uint64_t* primal;
  uint8_t* level;
  uint64_t capacity;
  __device__ void operator()(uint64_t i, unsigned long long v, unsigned long long ex) const {
    if (!v || ex >= capacity) return;
    const uint64_t k = keys[i];
    uint8_t lv = levels[i];
    for (uint64_t j = i; j > 0 && keys[j - 1] == k; --j)
      if (levels[j - 1] > lv) lv = levels[j - 1];
    primal[ex] = k;
    level[ex] = lv;
  }
};

// Whether the nodes of all depths have found room.
__device__ __forceinline__ bool tree_fits(const LhmcTree& T) {
  uint64_t n = 0;
  for (int d = 0; d <= T.d1; ++d) n += T.ctl[kLhmcCount + d];
  return n <= T.cap;
}

// ---- 3. dual cubes ----------------------------------------------------------
// kLevels: a vertex's corners are nodes of its own level at most
// (C.primal_level).  On the bit lattice that level needs no record: levels are
// depths there but for the origin's node of each depth (kLhmcDenseDepth is
// below the depths with more such keys), so no leaf that touches a vertex is
// deeper than the deepest that marks it, and the descents end at leaves.
template <bool kLevels>
__global__ __launch_bounds__(kTile) void k_cubes(LhmcTree T, LhmcCubes C) {
  __shared__ TileShared S;
  const uint64_t n = T.ctl[kLhmcPrimal + 1];
  if (!tree_fits(T) || n > C.primal_capacity) return;
  const uint64_t n_tiles = (n + kTile - 1) / kTile;
  uint64_t tile;
  for (bool more = true; next_tile(&T.ctl[kLhmcCubes], n_tiles, S, more, &tile); more = false) {
    const uint64_t p = tile * kTile + threadIdx.x;
    uint32_t cube = 0;
    uint32_t node[8];
    if (p < n) {
      const uint64_t key = C.primal[p];
      const int lv = kLevels ? C.primal_level[p] : T.d1;
      uint64_t m[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        constexpr unsigned kRemap[8] = {2, 3, 1, 0, 6, 7, 5, 4};  // marching_cubes_tables.rs:29
        m[i] = dual_vertex(key, lv, kRemap[i]);
        // depths 0 and 1 always refine: the descent starts among the 64 of depth 2
        node[i] = 9 + (static_cast<uint32_t>(m[i] >> (3 * (lv - 2))) & 63u);
      }
      for (int t = lv - 3; t >= 0; --t) {  // implicit_octree.rs:87-96, from above
        bool more = false;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const uint32_t child = T.child[node[i]];
          if (child == kLhmcLeaf) continue;
          node[i] = child + (static_cast<uint32_t>(m[i] >> (3 * t)) & 7u);
          more = true;
        }
        if (!more) break;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (!(T.values[node[i]] > 0.0f)) cube |= 1u << i;  // classify_corners
    }
    const uint32_t tri = p < n ? c_lt.tri_count[cube] : 0;
    unsigned long long upto;
    const unsigned long long ex =
        scan_tile(tri ? (1ull << 32) | tri : 0ull, tile, C.slot, &T.ctl[kLhmcErr], S, &upto);
    const uint64_t a = ex >> 32;
    if (tri && a < C.capacity) {
      uint4* dst = reinterpret_cast<uint4*>(C.corner + 8 * a);
      dst[0] = make_uint4(node[0], node[1], node[2], node[3]);
      dst[1] = make_uint4(node[4], node[5], node[6], node[7]);
      C.cube_case[a] = static_cast<uint8_t>(cube);
      C.tri_first[a] = static_cast<uint32_t>(ex);
    }
    if (tile + 1 == n_tiles && threadIdx.x == 0) T.ctl[kLhmcCubes + 1] = upto;
  }
}

// ---- 4. ownership -----------------------------------------------------------
// The listed cubes, none if some buffer so far was too small; and the table
// for their edges, sized by their triangles (at most three edges each).
__device__ __forceinline__ uint32_t listed_cubes(const LhmcTree& N, const LhmcCubes& C) {
  const uint64_t n = N.ctl[kLhmcCubes + 1] >> 32;
  return !tree_fits(N) || N.ctl[kLhmcPrimal + 1] > C.primal_capacity || n > C.capacity || lhmc_table_size(N.ctl[kLhmcCubes + 1]) > C.table_capacity
             ? 0
             : static_cast<uint32_t>(n);
}
__device__ __forceinline__ uint64_t table_mask(const LhmcTree& N) {
  return lhmc_table_size(N.ctl[kLhmcCubes + 1]) - 1;
}

// Sixteen lanes a cube, one an edge (four idle).  The owner of an edge is the
// first cube that lists it, and its first listing there (two edges of a cube
// are the same edge where corners coincide): the least of 16 * cube + order.
__global__ __launch_bounds__(256) void k_owner(LhmcTree N, LhmcCubes C, LhmcEdgeTable T) {
  const uint32_t n = listed_cubes(N, C);
  T.mask = table_mask(N);
  const int e = static_cast<int>(threadIdx.x & 15);
  for (uint32_t a = (blockIdx.x * 256 + threadIdx.x) >> 4; a < n; a += gridDim.x * 16) {
    const uint32_t cube = C.cube_case[a];
    if (e >= 12 || !(c_lt.edge_mask[cube] >> e & 1)) continue;
    uint64_t h = table_insert(T, edge_key(C.corner + 8 * static_cast<uint64_t>(a), e));
    if (h == ~0ull) {
      atomicOr(&N.ctl[kLhmcErr], kLhmcErrTable);
      h = 0;
    }
    C.edge_slot[12 * static_cast<uint64_t>(a) + e] = static_cast<uint32_t>(h);
    const uint32_t mine = 16 * a + __popc(static_cast<unsigned>(c_lt.before[cube][e]));
    if (T.owner[h] > mine) atomicMin(&T.owner[h], mine);
  }
}

// Counts the owned edges of 256 cubes a workgroup (four at a time a wavefront),
// scans the counts, and writes the owned edges' ids and crossings.
constexpr int kOwnCubes = 256;

__global__ __launch_bounds__(kTile) void k_own(LhmcTree N, LhmcCubes C, LhmcEdgeTable T,
                                               float* __restrict__ vertices, uint64_t vcap) {
  __shared__ TileShared S;
  __shared__ uint32_t s_count[kTileWaves];
  const uint32_t n = listed_cubes(N, C);
  const uint64_t n_tiles = (static_cast<uint64_t>(n) + kOwnCubes - 1) / kOwnCubes;
  const int lane = __lane_id(), wv = threadIdx.x >> 6, e = lane & 15;
  uint64_t tile;
  for (bool more = true; next_tile(&N.ctl[kLhmcOwn], n_tiles, S, more, &tile); more = false) {
    const uint64_t a0 = kOwnCubes * tile + 16 * wv + (lane >> 4);
    uint64_t own[4];
    uint32_t slot[4], first[4];
    F3 at[4];
    uint32_t count = 0;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const uint64_t a = a0 + 4 * r;
      const uint32_t cube = a < n ? C.cube_case[a] : 0;
      bool mine = false;
      slot[r] = 0;
      uint32_t before = 0;
      if (e < 12 && (c_lt.edge_mask[cube] >> e & 1)) {
        slot[r] = C.edge_slot[12 * a + e];
        before = c_lt.before[cube][e];
        mine = T.owner[slot[r]] == 16 * static_cast<uint32_t>(a) + __popc(before);
      }
      own[r] = __ballot(mine);
      // ids run cube by cube, and in a cube by first listing
      const uint32_t cubes = static_cast<uint32_t>(own[r] >> (lane & 48)) & 0xFFFFu;
      first[r] = count + static_cast<uint32_t>(__popcll(own[r] & ((1ull << (lane & 48)) - 1))) +
                 __popc(cubes & before);
      count += static_cast<uint32_t>(__popcll(own[r]));
    }
    if (lane == 0) s_count[wv] = count;
    // The crossings, while the counts are on their way.
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (!(own[r] >> lane & 1)) continue;
      // find_edge_crossings (marching_cubes_impl.rs:39-56) for local edge e
      const uint64_t a = a0 + 4 * r;
      const uint32_t ia = C.corner[8 * a + tables::kEdgeCorners[e][0]];
      const uint32_t ib = C.corner[8 * a + tables::kEdgeCorners[e][1]];
      const float va = N.values[ia], vb = N.values[ib];
      const uint64_t ka = N.keys[ia], kb = N.keys[ib];
      const F3 pa = center_of(ka, level_of(N.split, ka)), pb = center_of(kb, level_of(N.split, kb));
      const float delta = vb - va;
      const float t = (delta == 0.0f) ? 0.5f : -va / delta;
      const float s = 1.0f - t;
      at[r] = {pa.x * s + pb.x * t, pa.y * s + pb.y * t, pa.z * s + pb.z * t};
    }
    __syncthreads();
    if (wv == 0) {
      uint32_t total = 0;
      for (int w = 0; w < kTileWaves; ++w) total += s_count[w];
      const unsigned long long prefix =
          scan::look_back(tile, total, C.own_slot, &N.ctl[kLhmcErr]);
      if (lane == 0) {
        S.prefix = prefix;
        if (tile + 1 == n_tiles) N.ctl[kLhmcOwn + 1] = prefix + total;
      }
    }
    __syncthreads();
    uint64_t base = S.prefix;
    for (int w = 0; w < wv; ++w) base += s_count[w];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (!(own[r] >> lane & 1)) continue;
      const uint64_t id = base + first[r];
      T.id[slot[r]] = static_cast<uint32_t>(id);
      if (id >= vcap) continue;
      vertices[3 * id + 0] = at[r].x;
      vertices[3 * id + 1] = at[r].y;
      vertices[3 * id + 2] = at[r].z;
    }
    __syncthreads();  // s_count
  }
}

// ---- 5. emit ----------------------------------------------------------------
// Sixteen lanes a cube, one an index (at most fifteen).
__global__ __launch_bounds__(256) void k_indices(LhmcTree N, LhmcCubes C, LhmcEdgeTable T,
                                                 uint32_t* __restrict__ indices, uint64_t icap) {
  const uint32_t n = listed_cubes(N, C);
  const int j = static_cast<int>(threadIdx.x & 15);
  for (uint32_t a = (blockIdx.x * 256 + threadIdx.x) >> 4; a < n; a += gridDim.x * 16) {
    const uint32_t cube = C.cube_case[a];
    if (j >= 3 * c_lt.tri_count[cube]) continue;
    const uint64_t at = 3 * static_cast<uint64_t>(C.tri_first[a]) + j;
    if (at < icap)
      indices[at] = T.id[C.edge_slot[12 * static_cast<uint64_t>(a) + c_lt.tri[cube][j]]];
  }
}

__global__ __launch_bounds__(256) void k_table_clear(LhmcTree N, LhmcCubes C, LhmcEdgeTable T) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const uint32_t n = listed_cubes(N, C);
  if (i0 < 2) N.ctl[kLhmcOwn + i0] = 0ull;
  if (n == 0) return;
  const uint64_t mask = table_mask(N);
  for (uint64_t i = i0; i <= mask; i += stride) {
    T.keys[i] = kEmpty;
    T.owner[i] = 0xffffffffu;
  }
  for (uint64_t i = i0; i <= n / kOwnCubes; i += stride) C.own_slot[i] = 0ull;
}

__global__ __launch_bounds__(256) void k_clear(unsigned long long* ctl, uint64_t n_ctl,
                                               unsigned long long* slot, uint64_t n_slots,
                                               uint4* bits, uint64_t n_bits) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const uint64_t i0 = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (uint64_t i = i0; i < n_ctl; i += stride) ctl[i] = 0ull;
  for (uint64_t i = i0; i < n_slots; i += stride) slot[i] = 0ull;
  for (uint64_t i = i0; i < n_bits; i += stride) bits[i] = make_uint4(0, 0, 0, 0);
}

__global__ __launch_bounds__(256) void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride)
    p[i] = v;
}

unsigned grid_of(uint64_t n, uint64_t cap = 16384) {
  uint64_t b = (n + 255) / 256;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return static_cast<unsigned>(b);
}

uint64_t tiles_of(uint64_t n) { return (n + kTile - 1) / kTile; }

// Workgroups of a launch over tiles, whose number may be known to the device
// only: enough to fill the chip, no more than the buffers could need.
unsigned tile_grid(uint64_t most) {
  const uint64_t b = tiles_of(most);
  return static_cast<unsigned>(b < 1 ? 1 : b > 512 ? 512 : b);
}

hipError_t clear_scan(unsigned long long* ctl, unsigned long long* slot, uint64_t n_slots,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_clear, dim3(grid_of(n_slots, 2048)), dim3(256), 0, s, ctl, uint64_t{2}, slot,
                     n_slots, static_cast<uint4*>(nullptr), uint64_t{0});
  return hipGetLastError();
}

}  // namespace

uint64_t lhmc_primal_slots(int d1) {
  return tiles_of((1ull << (3 * d1)) / 64);
}

hipError_t launch_lhmc_clear(const LhmcTree& T, unsigned long long* slot, uint64_t n_slots,
                             hipStream_t s) {
  const uint64_t n_bits = T.bits ? (1ull << (3 * T.d1)) / 128 : 0;
  hipLaunchKernelGGL(k_clear, dim3(grid_of(n_bits > n_slots ? n_bits : n_slots, 2048)), dim3(256),
                     0, s, T.ctl, static_cast<uint64_t>(kLhmcCtlWords), slot, n_slots,
                     reinterpret_cast<uint4*>(T.bits), n_bits);
  return hipGetLastError();
}

hipError_t launch_lhmc_levels(const LhmcTree& T, const ProgramKind& kind, hipStream_t s) {
  const auto top = !kind.bounded ? k_top<0> : kind.stack ? k_top<2> : k_top<1>;
  const auto few = !kind.bounded ? k_level<0, 1> : kind.stack ? k_level<2, 1> : k_level<1, 1>;
  const auto many = !kind.bounded ? k_level<0, 4> : kind.stack ? k_level<2, 4> : k_level<1, 4>;
  hipLaunchKernelGGL(top, dim3(10), dim3(64), 0, s, T);
  for (int d = 4; d <= T.d1; ++d) {
    const uint64_t all = d < 12 ? 1ull << (3 * d) : T.cap, most = all < T.cap ? all : T.cap;
    if (d <= 5)
      hipLaunchKernelGGL(few, dim3(static_cast<unsigned>((most + 63) / 64)), dim3(64), 0, s, T, d);
    else
      hipLaunchKernelGGL(many, dim3(grid_of(most, 2048)), dim3(256), 0, s, T, d);
  }
  return hipGetLastError();
}

hipError_t launch_lhmc_primal(const LhmcTree& T, const LhmcCubes& C, unsigned long long* slot,
                              hipStream_t s) {
  const uint64_t n_words = (1ull << (3 * T.d1)) / 64;
  hipLaunchKernelGGL(k_list, dim3(tile_grid(n_words)), dim3(kTile), 0, s, T, C, n_words, slot);
  return hipGetLastError();
}

size_t lhmc_sort_temp_bytes(uint64_t n_pairs) {
  size_t bytes = 0;
  if (rocprim::radix_sort_pairs(nullptr, bytes, static_cast<const uint64_t*>(nullptr),
                                static_cast<uint64_t*>(nullptr),
                                static_cast<const uint8_t*>(nullptr),
                                static_cast<uint8_t*>(nullptr), static_cast<size_t>(n_pairs), 0,
                                64) != hipSuccess)
    return 0;
  return bytes;
}

hipError_t launch_lhmc_primal_sorted(const LhmcTree& T, int64_t n_nodes, uint64_t* pair_keys,
                                     uint8_t* pair_levels, uint64_t* sorted_keys,
                                     uint8_t* sorted_levels, void* temp, size_t temp_bytes,
                                     const LhmcCubes& C, unsigned long long* slot,
                                     hipStream_t s) {
  const uint64_t n_pairs = 8 * static_cast<uint64_t>(n_nodes);
  hipLaunchKernelGGL(k_primal_pairs, dim3(grid_of(static_cast<uint64_t>(n_nodes))), dim3(256), 0,
                     s, T, n_nodes, pair_keys, pair_levels);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  size_t bytes = temp_bytes;
  e = rocprim::radix_sort_pairs(temp, bytes, static_cast<const uint64_t*>(pair_keys), sorted_keys,
                                static_cast<const uint8_t*>(pair_levels), sorted_levels,
                                static_cast<size_t>(n_pairs), 0, 64, s);
  if (e != hipSuccess) return e;
  RunLoad load{sorted_keys, n_pairs};
  RunSink sink{sorted_keys, sorted_levels, C.primal, C.primal_level, C.primal_capacity};
  const scan::State st{slot, T.ctl + kLhmcPrimal, T.ctl + kLhmcErr};
  return scan::launch<scan::kItems>(n_pairs, load, sink, st, s);
}

void lhmc_level_splits(uint64_t split[kLhmcMaxLevels]) {
  // Morton::level, morton.rs:53-59 (the same libm log, f64)
  auto level = [](uint64_t a) {
    return a == 0 ? 0 : static_cast<int>(std::floor(std::log(static_cast<double>(a)) * 0.48089834696));
  };
  split[0] = 0;
  for (int d = 1; d < kLhmcMaxLevels; ++d) {
    const uint64_t base = 1ull << (3 * d);
    // the first offset k at which level(base + k) reaches d (level is
    // monotone in the key, and d at the depth's last key, offset hi)
    uint64_t lo = 0, hi = (d == 21) ? ~0ull - base : 7 * base - 1;
    while (lo < hi) {
      const uint64_t mid = lo + (hi - lo) / 2;
      if (level(base + mid) >= d) hi = mid;
      else lo = mid + 1;
    }
    split[d] = lo;
  }
}

hipError_t launch_lhmc_cubes_reset(const LhmcTree& T, const LhmcCubes& C, hipStream_t s) {
  return clear_scan(T.ctl + kLhmcCubes, C.slot, tiles_of(C.primal_capacity), s);
}

hipError_t launch_lhmc_cubes(const LhmcTree& T, const LhmcCubes& C, hipStream_t s) {
  const dim3 grid(tile_grid(C.primal_capacity));
  if (T.bits)
    hipLaunchKernelGGL(k_cubes<false>, grid, dim3(kTile), 0, s, T, C);
  else
    hipLaunchKernelGGL(k_cubes<true>, grid, dim3(kTile), 0, s, T, C);
  return hipGetLastError();
}

hipError_t launch_lhmc_own(const LhmcTree& N, const LhmcCubes& C, const LhmcEdgeTable& T,
                           float* vertices, uint64_t vcap, hipStream_t s) {
  const uint64_t lanes = 16 * C.capacity;
  hipLaunchKernelGGL(k_table_clear, dim3(grid_of(C.table_capacity, 1024)), dim3(256), 0, s, N, C,
                     T);
  hipLaunchKernelGGL(k_owner, dim3(grid_of(lanes, 4096)), dim3(256), 0, s, N, C, T);
  hipLaunchKernelGGL(k_own, dim3(tile_grid(C.capacity * (kTile / kOwnCubes))), dim3(kTile), 0, s, N,
                     C, T, vertices, vcap);
  return hipGetLastError();
}

hipError_t launch_lhmc_emit(const LhmcTree& N, const LhmcCubes& C, const LhmcEdgeTable& T,
                            uint32_t* indices, uint64_t icap, hipStream_t s) {
  hipLaunchKernelGGL(k_indices, dim3(grid_of(16 * C.capacity, 4096)), dim3(256), 0, s, N, C, T,
                     indices, icap);
  return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s) {
  hipLaunchKernelGGL(k_fill_u32, dim3(grid_of(n)), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace iso
