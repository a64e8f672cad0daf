// Sparse classification of program sources for gfx950 (MI355X).
//
// Marching cubes reads a sample's value only at the ends of an edge that
// crosses the surface, and everywhere else only its sign.  A workgroup of one,
// four or eight wavefronts takes a tile of 16^3 samples; its first wavefront, one
// lane for each of the tile's 64 bricks of 4^3, bounds the program over each
// brick's samples and their lattice neighbours (the box one sample wider on every
// side): where the bounds exclude zero, the sign of all of them is proven.  A
// crossing edge joins two neighbouring samples of different sign, so neither of
// them lies in a proven brick: the evaluated bricks hold every value that is
// read.  The same pass lists the operations that can change the program's value
// anywhere in the tile (sparse_eval.h), and the unproven bricks are evaluated
// over that list, dealt to the wavefronts, a sample of each of two or four bricks
// a lane.  Signs and values are the dense evaluation's, bit for bit.
//
// The sign words are row-aligned (each sample row starts a new word), so a
// tile's 16 samples of a row are one 16-bit store and no two tiles share a
// piece; the count and emit kernels take the row pitch from the CellSpace.
//
// Bound by instruction issue and the latency of one tile's chain (bounds of the
// tile, of its bricks, then its bricks' samples), not by memory: 64 spheres
// minus a torus at 257^3 evaluate 25,437 of 274,625 bricks over 8 operations
// each and take 44 us, where evaluating every sample took 617 us.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <cmath>

#include "mc_device.h"
#include "mc_kernels.h"
#include "sparse_eval.h"
#include "sparse_kernels.h"

namespace iso {

namespace {

using namespace mcd;

constexpr int kBricks = 64;      // bricks of a tile: 4 x 4 x 4
constexpr int kListCap = kTileListCap;
constexpr uint32_t kSparseXcds = 8;

// One lattice: its tiles x fastest.
struct SingleTiles {
  CellSpace C;
  __device__ __forceinline__ const CellSpace& at(uint32_t tile, uint32_t* local) const {
    *local = tile;
    return C;
  }
};

// A batch: the chunk that holds a tile is found by binary search of the
// chunks' first tiles.  The table is read through the constant address space:
// scalar loads, as the index is the same for the whole workgroup.
struct BatchTiles {
  const CellSpace* chunks;
  const uint32_t* tile_start;
  uint32_t n_chunks;
  __device__ __forceinline__ CellSpace at(uint32_t tile, uint32_t* local) const {
    using U32 = const uint32_t __attribute__((address_space(4)))*;
    const U32 first = (U32)(reinterpret_cast<uintptr_t>(tile_start));
    uint32_t lo = 0, hi = n_chunks;  // last chunk whose first tile <= tile
    while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) >> 1;
      if (first[mid] <= tile) lo = mid;
      else hi = mid;
    }
    *local = tile - first[lo];
    return load_space(chunks, lo);
  }
};

// W wavefronts per tile: one where tiles alone fill the chip, four or eight
// where a small lattice leaves it idle (the bricks of a tile are then spread
// over the SIMDs; the bounds are one wavefront's work either way).
//
// kSamples: for dual contouring, which takes no sign words but reads all
// samples, a dual value being half the sum of two opposite corners of a cell.
// A sample of a proven brick is 1 or -1 there.  A dual value is read for more
// than its sign only where its dual neighbour's differs, and the samples of
// both lie within two of any of them: the bounds are taken two samples wider,
// and from 1e-30 on where half a sample could round to zero.
//
// kDirected: Directed values (three floats a sample) and their signs.  A brick
// is proven where all components of all its samples, and its neighbours',
// have one sign (directed_interval), and the evaluated bricks again hold every
// value that is read, those of all corners of a mixed cell.
enum SparseMode : int { kSigns, kSamples, kDirected };

//
// kLong: the program may be longer than a list.  A tile whose list does not fit
// is then not bounded brick by brick (a chain as long as the program): all its
// bricks are evaluated, each wavefront bounding the operations for its own
// samples, 64 at a time (sdf_eval_near).  Whole extractions at 93^3, the program
// bounded and evaluated whole / near / the dense pass: 2040 smoothly joined
// spheres 3.87 / 0.44 / 0.68 ms, 2040 joined by minima 2.36 / 0.31 / 0.62; dual
// contouring of them 4.31 / 0.85 / 7.79 and 2.68 / 0.54 / 5.46.  Where the bounds
// of the tile leave nearly all operations in, the program is bounded and
// evaluated whole: 550 spheres that blend everywhere at 129^3 take 1.17 ms so,
// near 2.20.
template <class Tiles, int W, bool kStack, int kMode, bool kLong>
__global__ __launch_bounds__(64 * W) void k_signs_sparse(Tiles tiles, uint32_t n_tiles,
                                                         uint32_t group, ResetArgs R) {
  constexpr int kMargin = kMode == kSamples ? 2 : 1;  // neighbours in a brick's box
  constexpr int kTileCoords = kTileSide + 2 * kMargin;  // coordinates along an axis
  constexpr float kOutside = kMode == kSamples ? 1.0e-30f : 0.0f;
  __shared__ uint64_t s_sign[kBricks];  // sign bits of a brick's samples, x fastest
  __shared__ uint16_t s_list[kListCap];  // operations that matter in the tile
  __shared__ uint64_t s_mask[kListCap];  // and the bricks each of them matters in
  __shared__ float s_coord[3 * kTileCoords];
  __shared__ int s_len;
  __shared__ uint64_t s_todo;
  if (kMode != kSamples) reset_state(R);
  // Groups of consecutive tiles (a row's neighbours share lines of sign words
  // and values) go to one XCD, the groups round robin.
  const uint32_t q = blockIdx.x / kSparseXcds;
  const uint32_t tile =
      ((q / group) * kSparseXcds + blockIdx.x % kSparseXcds) * group + q % group;
  if (tile >= n_tiles) return;
  uint32_t local;
  const auto& C = tiles.at(tile, &local);
  const int32_t nx = static_cast<int32_t>(C.nx), ny = static_cast<int32_t>(C.ny),
                nz = static_cast<int32_t>(C.nz);
  const int32_t n[3] = {nx, ny, nz};
  const uint32_t ntx = static_cast<uint32_t>(nx + kTileSide - 1) >> kTileShift;
  const uint32_t nty = static_cast<uint32_t>(ny + kTileSide - 1) >> kTileShift;
  const uint32_t tz = local / (ntx * nty);
  const uint32_t tr = local - tz * (ntx * nty);
  const uint32_t ty = tr / ntx;
  const uint32_t tx = tr - ty * ntx;
  const int32_t s0[3] = {static_cast<int32_t>(tx << kTileShift),
                         static_cast<int32_t>(ty << kTileShift),
                         static_cast<int32_t>(tz << kTileShift)};
  const OpsPtr ops = as_constant(C.ops);
  const int n_ops = C.n_ops;
  const int lane = __lane_id();
  const int wv = W == 1 ? 0 : static_cast<int>(threadIdx.x >> 6);
  const int first = leading_scopes(ops, n_ops);

  if (wv == 0) {
    // Coordinates of the tile's samples and its neighbours' along each axis,
    // inside the program's leading scopes (past the lattice: the last sample's).
    if (lane < 3 * kTileCoords) {
      const int a = lane / kTileCoords;
      const int32_t na = a == 0 ? nx : a == 1 ? ny : nz;
      int32_t i = (a == 0 ? s0[0] : a == 1 ? s0[1] : s0[2]) + lane - kTileCoords * a - kMargin;
      i = i < 0 ? 0 : i < na ? i : na - 1;
      const float o = a == 0 ? C.origin[0] : a == 1 ? C.origin[1] : C.origin[2];
      const float d = a == 0 ? C.spacing[0] : a == 1 ? C.spacing[1] : C.spacing[2];
      float x = o + static_cast<float>(i) * d;  // as the dense kernels compute it
      for (int s = 0; s < first; ++s)
        x = x - (a == 0 ? ops[s].off[0] : a == 1 ? ops[s].off[1] : ops[s].off[2]);
      s_coord[lane] = x;
    }
    lds_barrier<1>();
    // The tile's bounds first: most tiles are proven here.
    float blo[3], bhi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const float c0 = s_coord[kTileCoords * a], c1 = s_coord[kTileCoords * a + kTileCoords - 1];
      blo[a] = fminf(c0, c1);
      bhi[a] = fmaxf(c0, c1);
    }
    float lo, hi;
    int len = bound_box<kStack, kMode == kDirected>(ops, first, n_ops, blo, bhi, s_list, kListCap, &lo, &hi);
    bool outside = lo > kOutside, inside = hi <= 0.0f;
    bool active = true;
    if (!outside && !inside) {
      // Then its bricks', each with its samples' neighbours.
      const int b[3] = {lane & 3, (lane >> 2) & 3, lane >> 4};
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        active = active && s0[a] + 4 * b[a] < n[a];
        const float c0 = s_coord[kTileCoords * a + 4 * b[a]];
        const float c1 = s_coord[kTileCoords * a + 4 * b[a] + 3 + 2 * kMargin];
        blo[a] = fminf(c0, c1);
        bhi[a] = fmaxf(c0, c1);
      }
      lds_barrier<1>();
      const bool fits = len <= kListCap;
      if (!kLong || fits || !prunes_near(len, n_ops)) {
        const int left = bound_lanes<kStack, kMode == kDirected>(
            ops, first, fits ? len : n_ops - first, blo, bhi, active, fits ? s_list : nullptr,
            s_mask, &lo, &hi);
        if (fits) len = left;
        outside = lo > kOutside;
        inside = hi <= 0.0f;
      }
    }
    s_sign[lane] = inside ? ~0ull : 0ull;
    const uint64_t todo = __ballot(active && !outside && !inside);
    if (lane == 0) {
      s_len = len;
      s_todo = todo;
    }
  }
  lds_barrier<W>();
  const int len = __builtin_amdgcn_readfirstlane(s_len);
  uint64_t todo;
  {
    const uint64_t t = s_todo;
    todo = static_cast<uint64_t>(static_cast<uint32_t>(
               __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t)))) |
           (static_cast<uint64_t>(static_cast<uint32_t>(
                __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(t >> 32))))
            << 32);
  }
  if (kMode == kSamples && ~todo) {
    // rows of sixteen samples, four a wavefront's store
    float* grid = const_cast<float*>(C.grid);
    for (int i = threadIdx.x; i < kTileSide * kTileSide * kTileSide; i += 64 * W) {
      const int x = i & 15, y = (i >> 4) & 15, z = i >> 8;
      const int b = (z >> 2) * 16 + (y & 12) + (x >> 2);
      if ((todo >> b & 1) || s0[0] + x >= nx || s0[1] + y >= ny || s0[2] + z >= nz) continue;
      grid[(static_cast<int64_t>(s0[2] + z) * ny + s0[1] + y) * nx + s0[0] + x] =
          s_sign[b] ? -1.0f : 1.0f;
    }
  }
  const uint16_t* list = len <= kListCap ? s_list : nullptr;
  const bool near = kLong && len > kListCap && prunes_near(len, n_ops);
  const int m = len <= kListCap ? len : n_ops - first;
  const int lx = lane & 3, ly = (lane >> 2) & 3, lz = lane >> 4;
  const bool full = s0[0] + kTileSide <= nx && s0[1] + kTileSide <= ny && s0[2] + kTileSide <= nz;
  // A lane's sample within its brick (lattices have less than 2^32 samples).
  const uint32_t within = (static_cast<uint32_t>(lz) * static_cast<uint32_t>(ny) +
                           static_cast<uint32_t>(ly)) * static_cast<uint32_t>(nx) +
                          static_cast<uint32_t>(lx);
  constexpr int kPoints = kStack ? 2 : 4;
  // kPoints bricks a round, the wavefronts' rounds interleaved.
  for (int k = 0; todo; ++k) {
    int brick[kPoints];
    uint32_t have = 0;
    uint64_t bricks = 0;
#pragma unroll
    for (int j = 0; j < kPoints; ++j) {
      brick[j] = j ? brick[0] : 0;
      if (todo) {
        brick[j] = static_cast<int>(__builtin_ctzll(todo));
        bricks |= todo & (0ull - todo);
        todo &= todo - 1;
        have |= 1u << j;
      }
    }
    if (W > 1 && (k & (W - 1)) != wv) continue;
    float p[kPoints][3], v[kPoints];
#pragma unroll
    for (int j = 0; j < kPoints; ++j) {
      const int b = brick[j];
      p[j][0] = s_coord[kMargin + 4 * (b & 3) + lx];
      p[j][1] = s_coord[kTileCoords + kMargin + (b & 12) + ly];
      p[j][2] = s_coord[2 * kTileCoords + kMargin + 4 * (b >> 4) + lz];
    }
    float d[kPoints][3];
    if constexpr (kMode == kDirected) {
      sdf_eval_vector_list<kPoints, kStack>(ops, first, list, s_mask, bricks, m, p, d);
#pragma unroll
      for (int j = 0; j < kPoints; ++j)  // Directed::is_positive, distance.rs:76-79
        v[j] = d[j][0] > 0.0f || d[j][1] > 0.0f || d[j][2] > 0.0f ? 1.0f : -1.0f;
    } else if (near) {
      // (outside the leading scopes, which it enters itself)
#pragma unroll
      for (int j = 0; j < kPoints; ++j) {
        const int b = brick[j];
        const int32_t at[3] = {s0[0] + 4 * (b & 3) + lx, s0[1] + (b & 12) + ly,
                               s0[2] + 4 * (b >> 4) + lz};
#pragma unroll
        for (int a = 0; a < 3; ++a)
          p[j][a] = C.origin[a] +
                    static_cast<float>(at[a] < n[a] ? at[a] : n[a] - 1) * C.spacing[a];
      }
      sdf_eval_near<kPoints, kStack>(ops, n_ops, lane_ops(ops, 0, n_ops), p, v);
    } else {
      sdf_eval_list<kPoints, kStack>(ops, first, list, s_mask, bricks, m, p, v);
    }
    uint64_t mine = 0;
#pragma unroll
    for (int j = 0; j < kPoints; ++j) {
      const int b = brick[j];
      const int32_t x0 = s0[0] + 4 * (b & 3), y0 = s0[1] + (b & 12), z0 = s0[2] + 4 * (b >> 4);
      const bool valid = full || (x0 + lx < nx && y0 + ly < ny && z0 + lz < nz);
      if (C.grid && valid && ((have >> j) & 1u)) {
        const int64_t s = (static_cast<int64_t>(z0) * ny + y0) * nx + x0 + within;
        float* at = const_cast<float*>(C.grid);
        if constexpr (kMode == kDirected) {
          at[3 * s + 0] = d[j][0];
          at[3 * s + 1] = d[j][1];
          at[3 * s + 2] = d[j][2];
        } else {
          at[s] = v[j];
        }
      }
      // classify_corners, distance.rs:52-54
      const uint64_t in = __ballot(valid && !(v[j] > 0.0f));
      if (lane == j) mine = in;
    }
    if (kMode == kSamples) continue;
    // (a spare point repeats the first brick)
    int slot = brick[0];
#pragma unroll
    for (int j = 1; j < kPoints; ++j) slot = lane == j ? brick[j] : slot;
    if (lane < kPoints) s_sign[slot] = mine;
  }
  if (kMode == kSamples) return;
  lds_barrier<W>();
  store_tile_signs(C, s_sign, s0, tx, threadIdx.x, 64 * W);
}

// Blocks that cover n tiles in groups dealt to the XCDs round robin.
uint64_t sparse_blocks(uint64_t n_tiles, uint64_t group) {
  const uint64_t per = kSparseXcds * group;
  return (n_tiles + per - 1) / per * per;
}

template <class Kernel, class Tiles>
hipError_t launch_tiles(Kernel kernel, int threads, const Tiles& tiles, int64_t n_tiles,
                        int64_t group, const ResetArgs& R, hipStream_t s) {
  const uint64_t blocks = sparse_blocks(static_cast<uint64_t>(n_tiles), static_cast<uint64_t>(group));
  if (blocks > 0x7fffffffull) return hipErrorInvalidValue;
  hipEvent_t a, z;
  if (take_launch_events(&a, &z))
    hipExtLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)),
                          dim3(static_cast<unsigned>(threads)), 0, s, a, z, 0, tiles,
                          static_cast<uint32_t>(n_tiles), static_cast<uint32_t>(group), R);
  else
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)),
                       dim3(static_cast<unsigned>(threads)), 0, s, tiles,
                       static_cast<uint32_t>(n_tiles), static_cast<uint32_t>(group), R);
  return hipGetLastError();
}

// Tiles from which one wavefront each is the better split, and up to which
// eight are: a chain's latency counts there.  Kernel times with one / four
// wavefronts a tile, 64 spheres minus a torus: 75 / 44 us at 257^3 (4913
// tiles), 87 / 83 at 385^3 (15625), 119 / 151 at 513^3 (35937).  Whole
// extractions with four / eight: 74 / 65 us at 129^3 (729 tiles), 76 / 78 at
// 193^3 (2197), 94 / 110 at 257^3; directed values of 32 boxes at 128^3 (512
// tiles) 94 / 72, dual contouring's samples there 40 / 35.
constexpr int64_t kManyTiles = 16384;
constexpr int64_t kFewTiles = 2048;

// Parameters and coordinates below this: no square or sum of squares of a
// primitive's operands overflows.
constexpr float kBoundedMagnitude = 1.0e15f;

bool small(float v) { return std::fabs(v) < kBoundedMagnitude; }  // false for NaN

}  // namespace

bool program_bounded(const DevOp* ops, int n_ops) {
  for (int i = 0; i < n_ops; ++i) {
    if (!small(ops[i].k)) return false;
    for (int j = 0; j < 4; ++j)
      if (!small(ops[i].prm[j]) || !small(ops[i].off[j])) return false;
  }
  return true;
}

bool lattice_bounded(const Lattice& L, float reach) {
  const int64_t n[3] = {L.nx, L.ny, L.nz};
  for (int a = 0; a < 3; ++a)
    if (!small(reach * L.origin[a]) || !small(reach * (L.spacing[a] * static_cast<float>(n[a]))))
      return false;
  return true;
}

int64_t tile_count(int64_t nx, int64_t ny, int64_t nz) {
  return ((nx + kTileSide - 1) >> kTileShift) * ((ny + kTileSide - 1) >> kTileShift) *
         ((nz + kTileSide - 1) >> kTileShift);
}

bool program_needs_stack(const DevOp* ops, int n_ops) {
  int pushes = 0;
  for (int i = 0; i < n_ops; ++i) pushes += ops[i].code <= kCylinder && ops[i].combine == kPush;
  return pushes > 1;
}

ProgramKind program_kind(const DevOp* ops, int n_ops) {
  ProgramKind K;
  K.bounded = program_bounded(ops, n_ops);
  K.stack = program_needs_stack(ops, n_ops);
  double off = 0.0, prm = 0.0;
  for (int i = 0; i < n_ops; ++i) {
    for (int a = 0; a < 3; ++a) off = std::fmax(off, std::fabs(static_cast<double>(ops[i].off[a])));
    double p = std::fabs(static_cast<double>(ops[i].k));
    for (int a = 0; a < 4; ++a) p += std::fabs(static_cast<double>(ops[i].prm[a]));
    prm = std::fmax(prm, p);
  }
  // a point moves by the open scopes' offsets and the primitive's own
  K.magnitude = static_cast<float>((kMaxPointStack + 1) * off + prm);
  return K;
}

namespace {

template <int kMode, bool kStack, bool kLong>
hipError_t launch_single_as(const SingleTiles& t, const Lattice& L, const ResetArgs& R,
                            hipStream_t s) {
  const int64_t n = tile_count(L.nx, L.ny, L.nz);
  const int64_t group = (L.nx + kTileSide - 1) >> kTileShift;
  if (n <= kFewTiles)
    return launch_tiles(k_signs_sparse<SingleTiles, 8, kStack, kMode, kLong>, 512, t, n, group, R, s);
  if constexpr (!kLong) {
    if (n >= kManyTiles)
      return launch_tiles(k_signs_sparse<SingleTiles, 1, kStack, kMode, false>, 64, t, n, group, R, s);
    return launch_tiles(k_signs_sparse<SingleTiles, 4, kStack, kMode, false>, 256, t, n, group, R, s);
  }
  return hipErrorInvalidValue;
}

template <int kMode>
hipError_t launch_single(const SingleTiles& t, bool stack, const Lattice& L, const ResetArgs& R,
                         hipStream_t s) {
  // (directed values have no evaluation near a wavefront's samples; tiles of
  // larger lattices span so little that lists fit)
  if constexpr (kMode != kDirected) {
    if (t.C.n_ops > kListCap && tile_count(L.nx, L.ny, L.nz) <= kFewTiles)
      return stack ? launch_single_as<kMode, true, true>(t, L, R, s)
                   : launch_single_as<kMode, false, true>(t, L, R, s);
  }
  return stack ? launch_single_as<kMode, true, false>(t, L, R, s)
               : launch_single_as<kMode, false, false>(t, L, R, s);
}

template <bool kStack, bool kLong>
hipError_t launch_batch_as(const BatchTiles& t, int64_t n_tiles, int64_t group, const ResetArgs& R,
                           hipStream_t s) {
  if (n_tiles >= kManyTiles)
    return launch_tiles(k_signs_sparse<BatchTiles, 1, kStack, kSigns, kLong>, 64, t, n_tiles, group,
                        R, s);
  return launch_tiles(k_signs_sparse<BatchTiles, 4, kStack, kSigns, kLong>, 256, t, n_tiles, group,
                      R, s);
}

ResetArgs reset_args(const McDims& D, const McBuffers& B) {
  ResetArgs R;
  R.signs = B.signs;
  R.n_words = D.n_sign_words;
  R.agg = B.agg;
  R.incl = B.incl;
  R.n_blocks = D.n_blocks;
  R.totals = B.totals;
  return R;
}

}  // namespace

hipError_t launch_signs_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                               const McDims& D, const McBuffers& B, float* values, hipStream_t s) {
  if (!ops || !B.signs || (D.sign_pitch & 63)) return hipErrorInvalidValue;
  const SingleTiles t{single_cell_space(L, D, B.signs, ops, n_ops, values, nullptr)};
  return launch_single<kSigns>(t, stack, L, reset_args(D, B), s);
}

hipError_t launch_directed_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                                  const McDims& D, const McBuffers& B, float* values,
                                  hipStream_t s) {
  if (!ops || !B.signs || !values || (D.sign_pitch & 63)) return hipErrorInvalidValue;
  const SingleTiles t{single_cell_space(L, D, B.signs, ops, n_ops, values, nullptr)};
  return launch_single<kDirected>(t, stack, L, reset_args(D, B), s);
}

hipError_t launch_samples_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                                 float* samples, hipStream_t s) {
  if (!ops || !samples) return hipErrorInvalidValue;
  const SingleTiles t{
      single_cell_space(L, mc_dims_pitched(L), nullptr, ops, n_ops, samples, nullptr)};
  return launch_single<kSamples>(t, stack, L, ResetArgs{}, s);
}

hipError_t launch_batch_signs_sparse(const BatchPlan& P, const McBuffers& B, int64_t n_blocks,
                                     hipStream_t s) {
  if (!P.sparse || !P.chunks || !P.tile_start) return hipErrorInvalidValue;
  const BatchTiles t{P.chunks, P.tile_start, P.n_chunks};
  ResetArgs R;
  R.signs = nullptr;
  R.n_words = 0;
  R.agg = B.agg;
  R.incl = B.incl;
  R.n_blocks = n_blocks;
  R.totals = B.totals;
  // About a row of a chunk's tiles.  Not a divisor of their usual numbers, 8, 27,
  // 64, 125: where a chunk of S cells has tiles of one sample at its ends, its
  // full ones would all go to the same half of the XCDs (1024 chunks of 17^3 over
  // four primitives with a value stack: signs 214 us by groups of 4, 137 by 8 or
  // 16, 85 by 7; over 31 without 487 / 350 / 217; of 65^3, 128 chunks, 133 / 133
  // / 144).
  constexpr int64_t kGroup = 7;
  if (P.long_programs)
    return P.stack ? launch_batch_as<true, true>(t, P.n_tiles, kGroup, R, s)
                   : launch_batch_as<false, true>(t, P.n_tiles, kGroup, R, s);
  return P.stack ? launch_batch_as<true, false>(t, P.n_tiles, kGroup, R, s)
                 : launch_batch_as<false, false>(t, P.n_tiles, kGroup, R, s);
}

}  // namespace iso
