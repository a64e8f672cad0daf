// Dual-contouring kernels for gfx950 (MI355X).
//
// DualContouring::extract (dual_contouring.rs:65-105) over
// DualGrid::traverse (traversal/dual_grid.rs:52-95) in four kernels before
// the marching-cubes pass over the dual lattice:
//   1. sample   the program at every primal lattice point (near the surface;
//               elsewhere its sign, launch_samples_sparse);
//   2. dual     one thread per primal cell: dual value
//               lerp(v0, v6, 0.5) = 0.5*v0 + 0.5*v6, and either the centre
//               lerp(c0, c6, 0.5) as dual vertex (cube index 0 or 255) or an
//               entry in the mixed-cell list and a mark at its eight corners;
//   3. normals  one wavefront per brick of 4^3 lattice points: the normal at
//               each marked point by central differences of the program
//               (source.rs:82-94), or with epsilon 0 the program's own
//               HermiteSource normals (implicit/*.rs sample_normal,
//               csg.rs:47-51), normalised or zero
//               (marching_cubes_impl.rs:58-69);
//   4. feature  one thread per listed mixed cell: TangentPlanes and the QEF
//               solve (feature/mod.rs:91-148, feature/qef.rs:36-68) with the
//               reference's f64 SVD.
// The lists have no order and their lengths stay in device memory: nothing
// waits for the host between the samples and the mesh.
// Every result is written to its cell's own slot.
#include <hip/hip_runtime.h>

#include "dc_kernels.h"
#include "mc_tables.h"
#include "qef_device.h"
#include "sparse_eval.h"

namespace iso {

namespace {

__global__ __launch_bounds__(256) void k_dc_sample(const DevOp* __restrict__ ops, int n_ops,
                                                   Lattice L, int64_t n_points,
                                                   float* __restrict__ out) {
  const uint32_t nx = static_cast<uint32_t>(L.nx);
  const uint32_t nxy = static_cast<uint32_t>(L.nx * L.ny);
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  // Whole wavefronts step together (the culled evaluator works on all 64
  // lanes); lanes past the end evaluate the last point and store nothing.
  const int lane = static_cast<int>(threadIdx.x & 63u);
  for (int64_t f0 = static_cast<int64_t>(blockIdx.x) * blockDim.x + (threadIdx.x & ~63u);
       f0 < n_points; f0 += stride) {
    const int64_t f = f0 + lane;
    const uint32_t ff = static_cast<uint32_t>(f < n_points ? f : n_points - 1);
    const uint32_t z = ff / nxy;
    const uint32_t r = ff - z * nxy;
    const uint32_t y = r / nx;
    const uint32_t x = r - y * nx;
    const float v = sdf_eval_culled(ops, n_ops, lattice_coord(L, 0, x), lattice_coord(L, 1, y),
                                    lattice_coord(L, 2, z));
    if (f < n_points) out[f] = v;
  }
}

__global__ __launch_bounds__(256) void k_dc_clear(uint4* __restrict__ marks, uint64_t n,
                                                  unsigned long long* __restrict__ counters) {
  if (blockIdx.x == 0 && threadIdx.x < kDcSlots) counters[threadIdx.x] = 0ull;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * 256;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride)
    marks[i] = make_uint4(0, 0, 0, 0);
}

// Marks are kept by bricks of 4^3 lattice points, 64 bytes each.
__device__ __forceinline__ uint64_t mark_at(const DcBricks& K, uint32_t x, uint32_t y, uint32_t z) {
  const uint64_t brick = (static_cast<uint64_t>(z >> 2) * K.ny + (y >> 2)) * K.nx + (x >> 2);
  return 64 * brick + 16 * (z & 3) + 4 * (y & 3) + (x & 3);
}

// Thread per primal cell (coalesced): dual values, centres, and the mixed
// cells.  A workgroup's mixed cells go to the segment of the list that its
// index names, as kDcSegments counters in lines of their own: one for all of
// them would be a queue of atomics as long as the pass.
__global__ __launch_bounds__(kDcThreads) void k_dc_dual(Lattice L, uint64_t n_cells, DcBuffers B,
                                                        DcBricks K) {
  __shared__ uint32_t s_wave[kDcThreads / 64];
  __shared__ uint32_t s_first;
  const uint64_t c = static_cast<uint64_t>(blockIdx.x) * kDcThreads + threadIdx.x;
  bool mixed = false;
  if (c < n_cells) {
    const int64_t nx = L.nx, ny = L.ny;
    const uint32_t cnx = static_cast<uint32_t>(nx - 1);
    const uint32_t cnxy = static_cast<uint32_t>((nx - 1) * (ny - 1));
    const uint32_t cc = static_cast<uint32_t>(c);
    const uint32_t z = cc / cnxy;
    const uint32_t r = cc - z * cnxy;
    const uint32_t y = r / cnx;
    const uint32_t x = r - y * cnx;
    float v[8];
    uint32_t cube = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t px = x + tables::kCorner[i][0], py = y + tables::kCorner[i][1],
                    pz = z + tables::kCorner[i][2];
      v[i] = B.samples[(pz * ny + py) * nx + px];
      if (!(v[i] > 0.0f)) cube |= 1u << i;  // classify_corners, distance.rs:52-54
    }
    // Signed::lerp (distance.rs:56-58) with factor 0.5: (1 - 0.5) * a + 0.5 * b
    B.dual_values[c] = 0.5f * v[0] + 0.5f * v[6];
    mixed = cube != 0u && cube != 255u;
    if (!mixed) {
      // Vec3::lerp (vector.rs:325-333) of corners 0 and 6
      const float c0x = lattice_coord(L, 0, x), c0y = lattice_coord(L, 1, y),
                  c0z = lattice_coord(L, 2, z);
      const float c6x = lattice_coord(L, 0, x + 1), c6y = lattice_coord(L, 1, y + 1),
                  c6z = lattice_coord(L, 2, z + 1);
      B.dual_points[3 * c + 0] = 0.5f * c0x + 0.5f * c6x;
      B.dual_points[3 * c + 1] = 0.5f * c0y + 0.5f * c6y;
      B.dual_points[3 * c + 2] = 0.5f * c0z + 0.5f * c6z;
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        B.marks[mark_at(K, x + tables::kCorner[i][0], y + tables::kCorner[i][1],
                        z + tables::kCorner[i][2])] = 1;
    }
  }
  const uint64_t all = __ballot(mixed);
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  if (lane == 0) s_wave[wv] = static_cast<uint32_t>(__popcll(all));
  __syncthreads();
  uint32_t before = 0, total = 0;
#pragma unroll
  for (int i = 0; i < kDcThreads / 64; ++i) {
    if (i < wv) before += s_wave[i];
    total += s_wave[i];
  }
  if (total == 0) return;
  const uint32_t segment = blockIdx.x % kDcSegments;
  if (threadIdx.x == 0)
    s_first = static_cast<uint32_t>(
        atomicAdd(&B.counters[kDcMixed + kDcLine * segment], static_cast<unsigned long long>(total)));
  __syncthreads();
  if (mixed)
    B.mixed[dc_segment_room(n_cells) * segment + s_first + before +
            __popcll(all & ((1ull << lane) - 1))] = static_cast<uint32_t>(c);
}

// CentralDifference::sample_normal (source.rs:82-94) at p, or with eps 0
// the program's HermiteSource::sample_normal, then
// normalised().unwrap_or_default() (marching_cubes_impl.rs:63-67).
__device__ __forceinline__ qef::Vec3f central_normal(const DevOp* ops, int n_ops, float px,
                                                     float py, float pz, float eps) {
  if (eps == 0.0f) {
    float raw[3];
    sdf_eval_hermite(ops, n_ops, px, py, pz, raw);
    return qef::normalised_or_zero(qef::Vec3f{raw[0], raw[1], raw[2]});
  }
  const float vx = sdf_eval(ops, n_ops, px + eps, py + 0.0f, pz + 0.0f) -
                   sdf_eval(ops, n_ops, px - eps, py - 0.0f, pz - 0.0f);
  const float vy = sdf_eval(ops, n_ops, px + 0.0f, py + eps, pz + 0.0f) -
                   sdf_eval(ops, n_ops, px - 0.0f, py - eps, pz - 0.0f);
  const float vz = sdf_eval(ops, n_ops, px + 0.0f, py + 0.0f, pz + eps) -
                   sdf_eval(ops, n_ops, px - 0.0f, py - 0.0f, pz - eps);
  const float e2 = 2.0f * eps;
  return qef::normalised_or_zero(qef::Vec3f{vx / e2, vy / e2, vz / e2});
}

// CentralDifference::sample_normal (source.rs:82-94) as the normal sinks use
// it (extractor.rs:46-69,97-127): not normalised.
__global__ __launch_bounds__(256) void k_sample_normals(const DevOp* __restrict__ ops, int n_ops,
                                                        const float* __restrict__ pts, uint64_t n,
                                                        float eps, float* __restrict__ out) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float px = pts[3 * i], py = pts[3 * i + 1], pz = pts[3 * i + 2];
  const float vx = sdf_eval(ops, n_ops, px + eps, py + 0.0f, pz + 0.0f) -
                   sdf_eval(ops, n_ops, px - eps, py - 0.0f, pz - 0.0f);
  const float vy = sdf_eval(ops, n_ops, px + 0.0f, py + eps, pz + 0.0f) -
                   sdf_eval(ops, n_ops, px - 0.0f, py - eps, pz - 0.0f);
  const float vz = sdf_eval(ops, n_ops, px + 0.0f, py + 0.0f, pz + eps) -
                   sdf_eval(ops, n_ops, px - 0.0f, py - 0.0f, pz - eps);
  const float e2 = 2.0f * eps;
  out[3 * i + 0] = vx / e2;
  out[3 * i + 1] = vy / e2;
  out[3 * i + 2] = vz / e2;
}

// The normal at each marked lattice point of a brick of 4^3, 12 bytes at the
// point's place in the lattice.  kKind: 1 a bounded program without a stack, 2
// one with a stack: then the operations are bounded over the brick's marked
// points and only those that can change a value there are evaluated, at the six
// points of a central difference at once.  (The normals of a 128^3 lattice over
// 32 boxes: 43 us; listing the points by a scan and evaluating all 32 at each
// took 35 and 87.)  0: without sound bounds on the program, its culled
// evaluation one point after the other; kEach: nor on the points, each lane by
// itself (a brick has few marked points, and the lanes of the others idle).
constexpr int kEach = 3;
template <int kKind>
__global__ __launch_bounds__(256) void k_dc_normals(const DevOp* __restrict__ ops, int n_ops,
                                                    Lattice L, DcBricks K, float eps,
                                                    const uint8_t* __restrict__ marks,
                                                    float* __restrict__ normals) {
  const int lane = __lane_id();
  const uint64_t n = K.count(), stride = static_cast<uint64_t>(gridDim.x) * 4;
  for (uint64_t b = static_cast<uint64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6); b < n;
       b += stride) {
    const bool marked = marks[64 * b + lane] != 0;
    const uint64_t all = __ballot(marked);
    if (!all) continue;
    const uint32_t bz = static_cast<uint32_t>(b / (K.nx * K.ny));
    const uint32_t br = static_cast<uint32_t>(b - bz * (K.nx * K.ny));
    const uint32_t by = static_cast<uint32_t>(br / K.nx);
    const uint32_t bx = static_cast<uint32_t>(br - by * K.nx);
    // the other lanes take a marked point too
    const int at = marked ? lane : static_cast<int>(__builtin_ctzll(all));
    const uint32_t x = 4 * bx + (at & 3), y = 4 * by + ((at >> 2) & 3), z = 4 * bz + (at >> 4);
    const float px = lattice_coord(L, 0, x), py = lattice_coord(L, 1, y),
                pz = lattice_coord(L, 2, z);
    qef::Vec3f nrm;
    if (kKind == kEach || eps == 0.0f) {
      nrm = central_normal(ops, n_ops, px, py, pz, eps);
    } else {
      // the points of central_normal
      const float p[6][3] = {{px + eps, py + 0.0f, pz + 0.0f}, {px - eps, py - 0.0f, pz - 0.0f},
                             {px + 0.0f, py + eps, pz + 0.0f}, {px - 0.0f, py - eps, pz - 0.0f},
                             {px + 0.0f, py + 0.0f, pz + eps}, {px - 0.0f, py - 0.0f, pz - eps}};
      float v[6];
      if constexpr (kKind == 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] = sdf_eval_culled(ops, n_ops, p[k][0], p[k][1], p[k][2]);
      } else {
        const OpsPtr list = as_constant(ops);
        sdf_eval_near<6, kKind == 2>(list, n_ops, lane_ops(list, 0, n_ops), p, v);
      }
      const float e2 = 2.0f * eps;
      nrm = qef::normalised_or_zero(
          qef::Vec3f{(v[0] - v[1]) / e2, (v[2] - v[3]) / e2, (v[4] - v[5]) / e2});
    }
    if (!marked) continue;
    float* out = normals + 3 * ((static_cast<uint64_t>(z) * L.ny + y) * L.nx + x);
    out[0] = nrm.x;
    out[1] = nrm.y;
    out[2] = nrm.z;
  }
}

constexpr int kFeatureThreads = 128;

__global__ __launch_bounds__(kFeatureThreads) void k_dc_feature(
    Lattice L, uint64_t n_cells, DcBuffers B, const float* __restrict__ normals_at) {
  bool stalled = false;
  const uint32_t segment = blockIdx.x % kDcSegments;
  const uint64_t n_mixed = B.counters[kDcMixed + kDcLine * segment];
  const uint32_t* mixed = B.mixed + dc_segment_room(n_cells) * segment;
  const uint64_t stride = static_cast<uint64_t>(gridDim.x / kDcSegments) * kFeatureThreads;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x / kDcSegments) * kFeatureThreads + threadIdx.x;
       i < n_mixed; i += stride) {
    const uint32_t c = mixed[i];
    const uint32_t cnx = static_cast<uint32_t>(L.nx - 1);
    const uint32_t cnxy = static_cast<uint32_t>((L.nx - 1) * (L.ny - 1));
    const uint32_t z = c / cnxy;
    const uint32_t r = c - z * cnxy;
    const uint32_t y = r / cnx;
    const uint32_t x = r - y * cnx;
    qef::Vec3f corners[8], normals[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t px = x + tables::kCorner[k][0], py = y + tables::kCorner[k][1],
                     pz = z + tables::kCorner[k][2];
      corners[k] = {lattice_coord(L, 0, px), lattice_coord(L, 1, py), lattice_coord(L, 2, pz)};
      const float* q = normals_at + 3 * ((static_cast<uint64_t>(pz) * L.ny + py) * L.nx + px);
      normals[k] = {q[0], q[1], q[2]};
    }
    const qef::Vec3f p = qef::place_feature(corners, normals, &stalled);
    B.dual_points[3 * static_cast<uint64_t>(c) + 0] = p.x;
    B.dual_points[3 * static_cast<uint64_t>(c) + 1] = p.y;
    B.dual_points[3 * static_cast<uint64_t>(c) + 2] = p.z;
  }
  if (stalled) atomicOr(&B.counters[kDcStalled], 1ull);
}

}  // namespace

hipError_t launch_dc_sample(const DevOp* ops, int n_ops, const ProgramKind& kind,
                            const Lattice& L, const DcBuffers& B, hipStream_t s) {
  if (!ops || !B.samples || !B.counters || !B.marks) return hipErrorInvalidValue;
  const uint64_t marks = 4 * dc_bricks(L).count();
  uint64_t clear = (marks + 255) / 256;
  if (clear > 4096) clear = 4096;
  hipLaunchKernelGGL(k_dc_clear, dim3(static_cast<unsigned>(clear)), dim3(256), 0, s,
                     reinterpret_cast<uint4*>(B.marks), marks, B.counters);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (sparse_lattice(L, kind.bounded))
    return launch_samples_sparse(ops, n_ops, kind.stack, L, B.samples, s);
  const int64_t n = L.nx * L.ny * L.nz;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(k_dc_sample, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, ops, n_ops,
                     L, n, B.samples);
  return hipGetLastError();
}

hipError_t launch_dc_dual(const Lattice& L, const DcBuffers& B, hipStream_t s) {
  const uint64_t n_cells = static_cast<uint64_t>((L.nx - 1) * (L.ny - 1) * (L.nz - 1));
  if (n_cells == 0 || n_cells > 0xffffffffull || !B.marks || !B.mixed) return hipErrorInvalidValue;
  const uint64_t blocks = (n_cells + kDcThreads - 1) / kDcThreads;
  hipLaunchKernelGGL(k_dc_dual, dim3(static_cast<unsigned>(blocks)), dim3(kDcThreads), 0, s, L,
                     n_cells, B, dc_bricks(L));
  return hipGetLastError();
}

hipError_t launch_sample_normals(const DevOp* ops, int n_ops, const float* points, uint64_t n,
                                 float epsilon, float* normals, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (!ops || !points || !normals) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_sample_normals, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0,
                     s, ops, n_ops, points, n, epsilon, normals);
  return hipGetLastError();
}

hipError_t launch_dc_normals(const DevOp* ops, int n_ops, const ProgramKind& kind,
                             const Lattice& L, float epsilon, const DcBuffers& B, float* normals,
                             hipStream_t s) {
  if (!ops || !normals) return hipErrorInvalidValue;
  const DcBricks K = dc_bricks(L);
  uint64_t blocks = (K.count() + 3) / 4;
  if (blocks > 65536) blocks = 65536;
  // (epsilon widens the points' box: bounds need it small as well)
  const bool near = lattice_bounded(L) && epsilon < 1.0e15f;
  const auto kernel = !near          ? k_dc_normals<kEach>
                      : !kind.bounded ? k_dc_normals<0>
                      : kind.stack    ? k_dc_normals<2>
                                      : k_dc_normals<1>;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, ops, n_ops, L, K,
                     epsilon, B.marks, normals);
  return hipGetLastError();
}

hipError_t launch_dc_feature(const Lattice& L, const DcBuffers& B, const float* normals,
                             hipStream_t s) {
  if (!normals) return hipErrorInvalidValue;
  const uint64_t n_cells = static_cast<uint64_t>((L.nx - 1) * (L.ny - 1) * (L.nz - 1));
  // A thread for every cell of a small lattice; of a large one a few percent
  // are mixed.
  uint64_t blocks = (dc_segment_room(n_cells) + kFeatureThreads - 1) / kFeatureThreads;
  if (blocks > 1024) blocks = 1024;
  hipLaunchKernelGGL(k_dc_feature, dim3(static_cast<unsigned>(blocks * kDcSegments)),
                     dim3(kFeatureThreads), 0, s, L, n_cells, B, normals);
  return hipGetLastError();
}

}  // namespace iso
