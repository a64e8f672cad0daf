// Launch interface of sparse program classification (sparse_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mc_kernels.h"
#include "sdf_program.h"

namespace iso {

// A tile: 16^3 samples, in 64 bricks of 4^3.
constexpr int kTileShift = 4;
constexpr int kTileSide = 1 << kTileShift;
constexpr int kTileListCap = 512;  // operations of a tile's list; a longer one is not kept

// Whether interval bounds of the program over this lattice are sound: every
// parameter and coordinate is finite and far from overflowing a square.
// `reach`: and so are points that many times as far out as the lattice's.
bool program_bounded(const DevOp* ops, int n_ops);
bool lattice_bounded(const Lattice& L, float reach = 1.0f);
// Whether the program holds values below the running one.
bool program_needs_stack(const DevOp* ops, int n_ops);

// What the kernels ask of a program.
struct ProgramKind {
  bool bounded = false;    // program_bounded
  bool stack = false;      // program_needs_stack
  float magnitude = 0.0f;  // bounds the offsets of its nested scopes, its parameters and widths
};
ProgramKind program_kind(const DevOp* ops, int n_ops);

// Whether a program lattice is classified sparsely: sound bounds, rows of at
// least one tile (narrower ones would leave most of a tile and of a sign word
// empty), and enough samples.  On a small lattice a tile spans many operands
// and few tiles run, so the dense pass is the faster one.  Whole extractions,
// dense / sparse, in us at 65^3, 81^3, 97^3 and 129^3:
//   marching cubes
//     64 spheres minus a torus         71 / 90    86 / 81   109 / 76   169 / 74
//     1000 smoothly joined spheres   309 / 1937 345 / 357  405 / 290  652 / 224
//     a sphere minus a torus           37 / 38    40 / 38    44 / 40    57 / 42
//   dual contouring, a box             87 / 94    91 / 94    95 / 97   125 / 116
//     32 boxes                        126 / 151  143 / 149  165 / 153  242 / 183
//     1000 smoothly joined spheres   464 / 2114 526 / 2112 653 / 624 1035 / 668
//   extended, a box                  129 / 134  131 / 132  136 / 136  146 / 135
//     32 boxes                       199 / 242  218 / 244  248 / 249  339 / 259
//     a torus (never proven)         108 / 118  113 / 121  118 / 127  130 / 144
constexpr int64_t kSparseMinPoints = 786432;  // 92^3
inline bool sparse_lattice(const Lattice& L, bool program_is_bounded) {
  return L.nx >= kTileSide && L.nx * L.ny * L.nz >= kSparseMinPoints && program_is_bounded &&
         lattice_bounded(L);
}

// Tiles of a lattice.
int64_t tile_count(int64_t nx, int64_t ny, int64_t nz);

// Whether a batch is classified sparsely, by the tiles and samples of its
// chunks (its programs and lattices bounded): a tile costs the bounds of its
// operations, a chain, however little of it the chunk fills.  Where more tiles
// than the chip holds at once are nearly empty, the flat pass over the samples
// does better: whole calls of 8192 chunks of 5^3, flat / sparse, over four
// primitives with a value stack 130 / 170 us, over two 95 / 113.  Chunks of 9^3
// fill enough (257 / 254), and 2048 chunks of 3^3 take 106 / 101.
constexpr int64_t kBatchManyTiles = 4096;
constexpr int64_t kBatchTileSamples = 256;
inline bool sparse_batch(int64_t tiles, int64_t samples) {
  return tiles < (int64_t(1) << 30) &&
         (tiles <= kBatchManyTiles || samples >= kBatchTileSamples * tiles);
}

// Program signs like launch_signs_program, from dims of mc_dims_pitched:
// bounds prove the sign of whole 4^3 bricks of samples, and only the bricks
// they cannot prove are evaluated (their samples go to `values` when it is
// not null).  Every lattice edge that crosses the surface has both its ends
// in evaluated bricks, and every sign is the evaluated program's.
// Program and lattice must be bounded; `stack`: program_needs_stack.
hipError_t launch_signs_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                               const McDims& D, const McBuffers& B, float* values, hipStream_t s);

// Directed signs and values like launch_signs_directed (3 floats a sample,
// those of the unproven bricks), from dims of mc_dims_pitched.
hipError_t launch_directed_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                                  const McDims& D, const McBuffers& B, float* values,
                                  hipStream_t s);

// Samples of a lattice for dual contouring: the program's value near the
// surface, and 1 or -1 at samples whose own and whose neighbours' dual values
// are only read for their sign.
hipError_t launch_samples_sparse(const DevOp* ops, int n_ops, bool stack, const Lattice& L,
                                 float* samples, hipStream_t s);

// The same for every chunk of a batch (P.sparse), and the extraction's state
// reset for n_blocks look-back words.
hipError_t launch_batch_signs_sparse(const BatchPlan& P, const McBuffers& B, int64_t n_blocks,
                                     hipStream_t s);

}  // namespace iso
