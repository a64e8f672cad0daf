// Launch interface of the dual-contouring kernels (host side).
//
// Dual contouring is marching cubes on the dual lattice: one dual point per
// primal cell, carrying the cell's dual value (the lerp of its corners 0 and
// 6) and its dual vertex (the cell centre, or for a mixed cell the feature
// point placed by the QEF).  These kernels build that lattice; the
// marching-cubes kernels then extract it with per-point positions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mc_kernels.h"
#include "sparse_kernels.h"
#include "sdf_program.h"

namespace iso {

// Slots of DcBuffers::counters.
constexpr int kDcSegments = 8;  // segments of the mixed-cell list
constexpr int kDcLine = 16;     // counters in lines of 128 bytes
enum : int {
  kDcStalled = 0,  // nonzero when a QEF's SVD hit the sweep bound
  kDcMixed = kDcLine,  // mixed primal cells listed in a segment, kDcLine apart
  kDcSlots = kDcLine * (1 + kDcSegments),
};

constexpr int kDcThreads = 1024;  // cells of a workgroup of the dual pass

// Entries of a list segment: the cells of every kDcSegments-th workgroup.
__host__ __device__ inline uint64_t dc_segment_room(uint64_t n_cells) {
  const uint64_t blocks = (n_cells + kDcThreads - 1) / kDcThreads;
  return (blocks + kDcSegments - 1) / kDcSegments * kDcThreads;
}

// The bricks of 4^3 lattice points that marks are kept by.
struct DcBricks {
  uint64_t nx, ny, nz;
  __host__ __device__ uint64_t count() const { return nx * ny * nz; }
};
inline DcBricks dc_bricks(const Lattice& L) {
  return {static_cast<uint64_t>(L.nx + 3) / 4, static_cast<uint64_t>(L.ny + 3) / 4,
          static_cast<uint64_t>(L.nz + 3) / 4};
}

struct DcBuffers {
  float* samples;       // primal lattice samples, nx*ny*nz
  float* dual_values;   // one per primal cell, z-major
  float* dual_points;   // 3 per primal cell
  uint32_t* mixed;      // mixed primal cells, kDcSegments * dc_segment_room(cells)
  uint8_t* marks;       // lattice points at a mixed cell, 64 per brick
  unsigned long long* counters;  // kDcSlots
};

// Samples the program over the primal lattice, and clears counters and marks.
hipError_t launch_dc_sample(const DevOp* ops, int n_ops, const ProgramKind& kind,
                            const Lattice& L, const DcBuffers& B, hipStream_t s);
// Dual values and centre dual vertices; lists the mixed cells and marks their
// corners.
hipError_t launch_dc_dual(const Lattice& L, const DcBuffers& B, hipStream_t s);
// CentralDifference::sample_normal of the program at n points (3 floats
// each, device), unnormalised, into normals (3 floats each, device).
hipError_t launch_sample_normals(const DevOp* ops, int n_ops, const float* points, uint64_t n,
                                 float epsilon, float* normals, hipStream_t s);
// The normal at each marked point (central differences of step epsilon, or the
// program's analytic normals when epsilon is 0, normalised), 3 floats at each
// lattice point.
hipError_t launch_dc_normals(const DevOp* ops, int n_ops, const ProgramKind& kind,
                             const Lattice& L, float epsilon, const DcBuffers& B, float* normals,
                             hipStream_t s);
// Feature points of the listed mixed cells from their corners' normals,
// TangentPlanes and the QEF solve, one thread per cell.
hipError_t launch_dc_feature(const Lattice& L, const DcBuffers& B, const float* normals,
                             hipStream_t s);

}  // namespace iso
