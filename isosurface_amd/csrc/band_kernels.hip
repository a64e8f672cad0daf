// Learned narrow-band extraction kernels for gfx950 (MI355X); see
// band_kernels.h for the method.  The network itself is in mlp_kernels.hip.
#include <hip/hip_runtime.h>

#include "band_kernels.h"
#include "mc_device.h"
#include <cmath>
#include <type_traits>

#include "sdf_eval.h"
#include "sparse_eval.h"
#include "sparse_kernels.h"

namespace iso {

namespace {

using namespace mcd;

constexpr int kCertifyListCap = 512;

struct BrickBox {
  int64_t lo[3], hi[3];  // sample range [lo, hi] per axis
};

__device__ __forceinline__ BrickBox brick_box(const Lattice& L, const BrickGrid& G, int64_t b) {
  const int64_t bx = b % G.nbx;
  const int64_t r = b / G.nbx;
  const int64_t by = r % G.nby;
  const int64_t bz = r / G.nby;
  const int64_t n[3] = {L.nx, L.ny, L.nz};
  const int64_t c[3] = {bx, by, bz};
  BrickBox B;
  for (int a = 0; a < 3; ++a) {
    B.lo[a] = static_cast<int64_t>(G.brick) * c[a];
    B.hi[a] = B.lo[a] + G.brick < n[a] - 1 ? B.lo[a] + G.brick : n[a] - 1;
  }
  return B;
}

__global__ __launch_bounds__(256) void k_brick_centres(Lattice L, BrickGrid G,
                                                       float* __restrict__ centres,
                                                       float* __restrict__ half_diag) {
  const int64_t b = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (b >= G.n) return;
  const BrickBox B = brick_box(L, G, b);
  // Every brick is tested with the half-diagonal of a full brick (bricks
  // cut by the lattice's far faces are smaller), so one calibration holds
  // for all of them.
  float d2 = 0.0f;
  for (int a = 0; a < 3; ++a) {
    const float mid = 0.5f * static_cast<float>(B.lo[a] + B.hi[a]);
    centres[3 * b + a] = L.origin[a] + mid * L.spacing[a];
    const float ext = static_cast<float>(G.brick) * L.spacing[a];
    d2 += ext * ext;
  }
  half_diag[b] = 0.5f * sqrtf(d2);
}

// Adds the number of lanes with `on` set to *counter (one atomic per wave).
__device__ __forceinline__ void count_lanes(bool on, unsigned long long* counter) {
  const uint64_t m = __ballot(on);
  if (on && __lane_id() == __builtin_ctzll(m))
    atomicAdd(counter, static_cast<unsigned long long>(__popcll(m)));
}

// Every program is 1-Lipschitz (exact primitive distances, min, max,
// negation, translation and the polynomial smooth minimum, whose gradient is
// a convex combination of its operands'), so a centre value farther from
// zero than the distance to any sample of the box, plus the f32 evaluation
// error at both, proves that every sample of the box has the centre's sign.
// `widen` bounds the distance between the computed centre and any computed
// sample position (the half-diagonal, with the f32 rounding of both
// positions, pos_slack); the evaluation's own bound E holds at every point
// within `widen` of the centre, so the sample's f32 value lies within
// v +- (widen + 2E) and the sign is proven when |v| exceeds that.
__device__ __forceinline__ uint8_t certify_at(const DevOp* __restrict__ ops, int n_ops, float x,
                                              float y, float z, float half_diag,
                                              float pos_slack) {
  const float widen = half_diag * (1.0f + kCertifyRelSlack) + pos_slack;
  float e;
  const float v = sdf_eval_bound(ops, n_ops, x, y, z, widen, &e);
  return fabsf(v) > widen + 2.0f * e + kCertifyAbsSlack
             ? static_cast<uint8_t>(kBrickProven | (!(v > 0.0f) ? kBrickInside : 0))
             : static_cast<uint8_t>(0);
}

__global__ __launch_bounds__(256) void k_coarse_certify(const DevOp* __restrict__ ops, int n_ops,
                                                        Lattice L, BrickGrid G,
                                                        uint8_t* __restrict__ coarse,
                                                        unsigned long long* certified,
                                                        float pos_slack) {
  const int64_t s = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  count_lanes(s < G.nc, certified);
  if (s >= G.nc) return;
  const int64_t sx = s % G.ncx;
  const int64_t r = s / G.ncx;
  const int64_t c[3] = {sx, r % G.ncy, r / G.ncy};
  const int64_t n[3] = {L.nx, L.ny, L.nz};
  const int64_t kSpan = static_cast<int64_t>(G.brick) * kCoarse;  // cells per edge
  float p[3];
  float d2 = 0.0f;
  for (int a = 0; a < 3; ++a) {
    // The closed sample box [lo, hi] holds every brick box of the super-brick.
    const int64_t lo = kSpan * c[a];
    const int64_t hi = lo + kSpan < n[a] - 1 ? lo + kSpan : n[a] - 1;
    p[a] = L.origin[a] + 0.5f * static_cast<float>(lo + hi) * L.spacing[a];
    const float ext = static_cast<float>(kSpan) * L.spacing[a];
    d2 += ext * ext;
  }
  coarse[s] = certify_at(ops, n_ops, p[0], p[1], p[2], 0.5f * sqrtf(d2), pos_slack);
}

// Brick proofs: one wavefront per super-brick, one lane per brick (4 x 4 x 4
// bricks, x fastest), so a wavefront either copies its super-brick's proof
// or evaluates all of its bricks' centres together.
__global__ __launch_bounds__(256) void k_brick_certify(const DevOp* __restrict__ ops, int n_ops,
                                                       BrickGrid G,
                                                       const uint8_t* __restrict__ coarse,
                                                       const float* __restrict__ centres,
                                                       const float* __restrict__ half_diag,
                                                       uint8_t* __restrict__ proof,
                                                       unsigned long long* certified,
                                                       float pos_slack) {
  static_assert(kCoarse * kCoarse * kCoarse == 64, "one lane per brick of a super-brick");
  const int lane = __lane_id();
  const int64_t s = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (s >= G.nc) return;  // uniform per wave
  const int64_t sx = s % G.ncx;
  const int64_t r = s / G.ncx;
  const int64_t bx = kCoarse * sx + lane % kCoarse;
  const int64_t by = kCoarse * (r % G.ncy) + (lane / kCoarse) % kCoarse;
  const int64_t bz = kCoarse * (r / G.ncy) + lane / (kCoarse * kCoarse);
  const bool live = bx < G.nbx && by < G.nby && bz < G.nbz;
  const int64_t b = (bz * G.nby + by) * G.nbx + bx;
  const uint8_t cf = coarse[s];
  const bool evaluate = live && !(cf & kBrickProven);
  count_lanes(evaluate, certified);
  uint8_t out = cf;
  if (evaluate) {
    out = certify_at(ops, n_ops, centres[3 * b], centres[3 * b + 1], centres[3 * b + 2],
                     half_diag[b], pos_slack);
  }
  if (live) proof[b] = out;
}

// k_brick_certify for bounded programs.  A wavefront evaluates its bricks'
// centres over the operations that matter in the box of the centres: the
// values are the whole program's, and so are the proofs.  The operations left
// out enter an evaluation's error bound only as one more operand of its
// maximum, so the bound lies between the one of the listed operations alone
// and the one that starts from the greatest bound of any operation in the box;
// where the two decide a brick differently, the wavefront evaluates the whole
// program after all.
template <bool kStack>
__global__ __launch_bounds__(256) void k_brick_certify_listed(
    const DevOp* __restrict__ dops, int n_ops, BrickGrid G, const uint8_t* __restrict__ coarse,
    const float* __restrict__ centres, const float* __restrict__ half_diag,
    uint8_t* __restrict__ proof, unsigned long long* certified, float pos_slack, float mag) {
  __shared__ uint16_t s_list[4][kCertifyListCap];
  const int lane = __lane_id();
  const int wv = static_cast<int>(threadIdx.x >> 6);
  const int64_t s = static_cast<int64_t>(blockIdx.x) * 4 + wv;
  if (s >= G.nc) return;  // uniform per wave
  const int64_t sx = s % G.ncx;
  const int64_t r = s / G.ncx;
  const int64_t bx = kCoarse * sx + lane % kCoarse;
  const int64_t by = kCoarse * (r % G.ncy) + (lane / kCoarse) % kCoarse;
  const int64_t bz = kCoarse * (r / G.ncy) + lane / (kCoarse * kCoarse);
  const bool live = bx < G.nbx && by < G.nby && bz < G.nbz;
  const int64_t b = (bz * G.nby + by) * G.nbx + bx;
  const uint8_t cf = coarse[s];
  if (cf & kBrickProven) {
    if (live) proof[b] = cf;
    return;
  }
  const uint64_t lives = __ballot(live);
  if (lane == 0)
    atomicAdd(certified + kCounterStride * (s % kCounterLines),
              static_cast<unsigned long long>(__popcll(lives)));
  const OpsPtr ops = as_constant(dops);
  float p[3], lo[3], hi[3], widen = 0.0f;
  if (live) widen = half_diag[b] * (1.0f + kCertifyRelSlack) + pos_slack;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    p[a] = live ? centres[3 * b + a] : 0.0f;
    lo[a] = wave_min(live ? p[a] : kNoBound);
    hi[a] = -wave_min(live ? -p[a] : kNoBound);
  }
  const float wide = -wave_min(-widen);
  float floor_e;
  const int len = certify_list(ops, n_ops, lo, hi, wide, mag, s_list[wv], kCertifyListCap, &floor_e);
  lds_barrier<1>();
  uint8_t out = 0;
  bool unsure = true;
  if (len <= kCertifyListCap) {
    float e0, e1;
    const float v =
        eval_bound_list<kStack>(ops, s_list[wv], len, p[0], p[1], p[2], widen, floor_e, &e0, &e1);
    const bool p0 = fabsf(v) > widen + 2.0f * e0 + kCertifyAbsSlack;
    const bool p1 = fabsf(v) > widen + 2.0f * e1 + kCertifyAbsSlack;
    unsure = p0 != p1;
    out = p1 ? static_cast<uint8_t>(kBrickProven | (!(v > 0.0f) ? kBrickInside : 0)) : uint8_t{0};
  }
  if (__ballot(live && unsure) && live)
    out = certify_at(dops, n_ops, p[0], p[1], p[2], half_diag[b], pos_slack);
  if (live) proof[b] = out;
}

// The bricks' band and inside flags, with the numbers of band bricks and of
// network culls that no proof allows.
__global__ __launch_bounds__(256) void k_brick_flags(
    uint64_t n, const float* __restrict__ pred, const float* __restrict__ half_diag,
    const uint8_t* __restrict__ proof, float margin, uint8_t* __restrict__ flags,
    unsigned long long* n_band, unsigned long long* overturned) {
  __shared__ uint32_t s_sum[2];
  uint32_t bands = 0, turned = 0;
  if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n;
       i += stride) {
    bool band = true, inside = false;
    if (pred) {
      const float p = pred[i];
      // A NaN prediction is never trusted: the brick stays in the band.
      band = !(fabsf(p) > half_diag[i] + margin);
      inside = !(p > 0.0f);
    }
    if (proof) {
      const uint8_t pf = proof[i];
      const bool proven = (pf & kBrickProven) != 0;
      turned += pred != nullptr && !band && !proven;
      band = !proven;
      inside = proven && (pf & kBrickInside) != 0;
    }
    flags[i] = static_cast<uint8_t>((band ? kBrickBand : 0) | (inside ? kBrickInside : 0));
    bands += band;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    bands += __shfl_xor(bands, d, 64);
    turned += __shfl_xor(turned, d, 64);
  }
  if (__lane_id() == 0) {
    atomicAdd(&s_sum[0], bands);
    atomicAdd(&s_sum[1], turned);
  }
  __syncthreads();
  const int line = kCounterStride * (blockIdx.x % kCounterLines);
  if (threadIdx.x == 0 && s_sum[0]) atomicAdd(n_band + line, static_cast<unsigned long long>(s_sum[0]));
  if (threadIdx.x == 1 && s_sum[1])
    atomicAdd(overturned + line, static_cast<unsigned long long>(s_sum[1]));
}

// Signs and exact samples of one 16^3-sample tile (sparse_kernels.h) of the
// band's lattice.  A sample is exact when a band brick's closed sample box
// holds it (up to eight bricks do); every other one takes its own brick's
// predicted sign.  The tile's exact samples are queued in LDS, the samples of
// a 4^3 block of samples together, so that whole wavefronts evaluate 256 of
// them at a time however few each block has; with sound bounds they are
// evaluated over the operations that matter in the tile and, of those, in the
// blocks that the 256 come from.  Row-aligned sign words, one 16-bit store a
// row.  kKind: 0 any program, 1 bounded without a stack, 2 bounded with one;
// of the first each wavefront skips by sdf_eval_culled what cannot change its own
// 64 samples.  Bound by instruction issue: 98.4 M samples of
// 1024 smoothly joined spheres at 1025^3 take 4.8 ms, where the flat background
// pass and a culled evaluation of the whole program took 19.2 ms.
constexpr int kTileBlocks = 64;
constexpr int kTileSamples = kTileSide * kTileSide * kTileSide;
constexpr int kBandListCap = kTileListCap;
constexpr int kBandCoords = kTileSide + 2;
constexpr int kBandWaves = 4;
// A program longer than a tile's list on a lattice of few tiles: a tile then
// spans much of the domain and its list seldom fits, so wavefronts that cull for
// themselves do better, and there are few of them: sixteen a tile.  The exact
// samples of 1000 smoothly joined spheres, by lists and four wavefronts a tile /
// culled by four / by sixteen: 2261 / 874 / 295 us at 33^3 (27 tiles), 418 / 927
// / 342 at 65^3 (125); at 129^3 (729) 204 / 785 by four.
constexpr int64_t kBandFewTiles = 128;
constexpr int kBandManyWaves = 16;

// kLong: a program longer than a list; where it does not fit in a tile, the
// wavefronts bound the operations for their own samples (sdf_eval_near): 1500
// spheres joined over a width of 0.1 at 93^3 take 2.37 ms a call, 5.40 whole.
template <int kKind, int W, bool kLong>
__global__ __launch_bounds__(64 * W) void k_band_tiles(
    CellSpace C, BrickGrid G, const uint8_t* __restrict__ flags, uint32_t n_tiles,
    unsigned long long* evaluated, ResetArgs R) {
  constexpr bool kStack = kKind == 2;
  __shared__ uint64_t s_sign[kTileBlocks];
  __shared__ uint64_t s_mask[kBandListCap];
  __shared__ uint64_t s_from[kTileSamples / 64];  // blocks that each 64 queue entries come from
  __shared__ uint16_t s_queue[kTileSamples];
  __shared__ uint16_t s_list[kBandListCap];
  __shared__ float s_coord[3 * kBandCoords];
  __shared__ uint8_t s_flag[125];
  __shared__ uint32_t s_n;
  __shared__ int s_len;
  reset_state(R);
  const uint32_t tile = blockIdx.x;
  if (tile >= n_tiles) return;
  const int32_t n[3] = {static_cast<int32_t>(C.nx), static_cast<int32_t>(C.ny),
                        static_cast<int32_t>(C.nz)};
  const int32_t nb[3] = {static_cast<int32_t>(G.nbx), static_cast<int32_t>(G.nby),
                         static_cast<int32_t>(G.nbz)};
  const uint32_t ntx = static_cast<uint32_t>(n[0] + kTileSide - 1) >> kTileShift;
  const uint32_t nty = static_cast<uint32_t>(n[1] + kTileSide - 1) >> kTileShift;
  const uint32_t tz = tile / (ntx * nty);
  const uint32_t tr = tile - tz * (ntx * nty);
  const uint32_t ty = tr / ntx;
  const uint32_t tx = tr - ty * ntx;
  const int32_t s0[3] = {static_cast<int32_t>(tx << kTileShift),
                         static_cast<int32_t>(ty << kTileShift),
                         static_cast<int32_t>(tz << kTileShift)};
  const int lane = __lane_id();
  const int wv = static_cast<int>(threadIdx.x >> 6);
  // Flags of the tile's bricks and the ones below them: at most 5 per axis,
  // entry 0 the brick below the tile's first.
  const int per = (kTileSide >> G.shift) + 1;
  bool any = false;
  if (static_cast<int>(threadIdx.x) < per * per * per) {
    const int q[3] = {static_cast<int>(threadIdx.x) % per,
                      static_cast<int>(threadIdx.x) / per % per,
                      static_cast<int>(threadIdx.x) / (per * per)};
    int32_t b[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      b[a] = (s0[a] >> G.shift) - 1 + q[a];
      b[a] = b[a] < 0 ? 0 : b[a] < nb[a] ? b[a] : nb[a] - 1;
    }
    const uint8_t f = flags[(static_cast<int64_t>(b[2]) * G.nby + b[1]) * G.nbx + b[0]];
    s_flag[threadIdx.x] = f;
    any = (f & kBrickBand) != 0;
  }
  if (threadIdx.x == 0) s_n = 0;
  if (threadIdx.x < kTileSamples / 64) s_from[threadIdx.x] = 0ull;
  const bool work = __syncthreads_or(any) != 0;

  // Lane b looks at block b (4^3 samples): bit k of its word says whether the
  // brick that holds a sample on the block's low faces along the axes of k is
  // in the band (bit 0: the block's own brick), bit 8 the own brick's sign.
  uint32_t around = 0;
  {
    int own[3], low[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int32_t s = s0[a] + (a == 0 ? 4 * (lane & 3) : a == 1 ? lane & 12 : 4 * (lane >> 4));
      const int32_t first = (s0[a] >> G.shift) - 1;
      const int32_t b = s >> G.shift;
      // (blocks past the lattice: any entry)
      own[a] = (b < nb[a] ? b : nb[a] - 1) - first;
      if (own[a] < 0) own[a] = 0;
      low[a] = (s & (G.brick - 1)) == 0 && s > 0 && b <= nb[a] ? b - 1 - first : own[a];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint8_t f = s_flag[((k & 4 ? low[2] : own[2]) * per + (k & 2 ? low[1] : own[1])) * per +
                               (k & 1 ? low[0] : own[0])];
      around |= (f & kBrickBand ? 1u : 0u) << k;
      if (k == 0) around |= (f & kBrickInside ? 1u : 0u) << 8;
    }
  }
  if (!work) {
    if (wv == 0) s_sign[lane] = around & 256u ? ~0ull : 0ull;
    __syncthreads();
    store_tile_signs(C, s_sign, s0, tx, threadIdx.x, 64 * W);
    return;
  }
  // Each block, a wavefront at a time: signs of the samples that are not
  // exact, the others queued.
  const int l[3] = {lane & 3, (lane >> 2) & 3, lane >> 4};
  uint32_t held = 0;  // the bits of a block's word whose bricks hold this lane's sample
#pragma unroll
  for (int k = 0; k < 8; ++k)
    held |= (!(k & 1) || l[0] == 0) && (!(k & 2) || l[1] == 0) && (!(k & 4) || l[2] == 0) ? 1u << k : 0u;
  const bool full =
      s0[0] + kTileSide <= n[0] && s0[1] + kTileSide <= n[1] && s0[2] + kTileSide <= n[2];
  for (int blk = wv; blk < kTileBlocks; blk += W) {
    const uint32_t w = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(around), blk));
    const bool valid = full || (s0[0] + 4 * (blk & 3) + l[0] < n[0] &&
                                s0[1] + (blk & 12) + l[1] < n[1] &&
                                s0[2] + 4 * (blk >> 4) + l[2] < n[2]);
    const bool exact = valid && (w & held & 255u) != 0u;
    const uint64_t m = __ballot(exact);
    uint32_t at = 0;
    if (lane == 0) {
      s_sign[blk] = w & 256u ? ~m : 0ull;
      if (m) {
        const uint32_t cnt = static_cast<uint32_t>(__popcll(m));
        at = atomicAdd(&s_n, cnt);
        atomicOr(reinterpret_cast<unsigned long long*>(&s_from[at >> 6]), 1ull << blk);
        atomicOr(reinterpret_cast<unsigned long long*>(&s_from[(at + cnt - 1) >> 6]), 1ull << blk);
      }
    }
    if (m == 0ull) continue;
    at = __builtin_amdgcn_readfirstlane(at);
    if (exact)
      s_queue[at + static_cast<uint32_t>(__popcll(m & ((1ull << lane) - 1ull)))] =
          static_cast<uint16_t>(blk * 64 + lane);
  }
  __syncthreads();
  const uint32_t total = __builtin_amdgcn_readfirstlane(s_n);
  if (total) {
    const OpsPtr ops = as_constant(C.ops);
    const int n_ops = C.n_ops;
    const int first = kKind ? leading_scopes(ops, n_ops) : 0;
    if (wv == 0) {
      if (lane < 3 * kBandCoords) {
        const int a = lane / kBandCoords;
        const int32_t na = a == 0 ? n[0] : a == 1 ? n[1] : n[2];
        int32_t i = (a == 0 ? s0[0] : a == 1 ? s0[1] : s0[2]) + lane - kBandCoords * a - 1;
        i = i < 0 ? 0 : i < na ? i : na - 1;
        const float org = a == 0 ? C.origin[0] : a == 1 ? C.origin[1] : C.origin[2];
        const float d = a == 0 ? C.spacing[0] : a == 1 ? C.spacing[1] : C.spacing[2];
        float x = org + static_cast<float>(i) * d;
        for (int s = 0; s < first; ++s)
          x = x - (a == 0 ? ops[s].off[0] : a == 1 ? ops[s].off[1] : ops[s].off[2]);
        s_coord[lane] = x;
      }
      lds_barrier<1>();
      int len = kBandListCap + 1;
      if constexpr (kKind != 0) {
        float blo[3], bhi[3], vlo, vhi;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
          const float c0 = s_coord[kBandCoords * a + 1], c1 = s_coord[kBandCoords * a + kTileSide];
          blo[a] = fminf(c0, c1);
          bhi[a] = fmaxf(c0, c1);
        }
        len = bound_box<kStack>(ops, first, n_ops, blo, bhi, s_list, kBandListCap, &vlo, &vhi);
        if (len <= kBandListCap) {
          const int b[3] = {lane & 3, (lane >> 2) & 3, lane >> 4};
          bool active = true;
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            active = active && s0[a] + 4 * b[a] < n[a];
            const float c0 = s_coord[kBandCoords * a + 1 + 4 * b[a]];
            const float c1 = s_coord[kBandCoords * a + 4 + 4 * b[a]];
            blo[a] = fminf(c0, c1);
            bhi[a] = fmaxf(c0, c1);
          }
          lds_barrier<1>();
          len = bound_lanes<kStack>(ops, first, len, blo, bhi, active, s_list, s_mask, &vlo, &vhi);
        }
      }
      if (lane == 0) s_len = len;
    }
    __syncthreads();
    const int len = __builtin_amdgcn_readfirstlane(s_len);
    const uint16_t* list = len <= kBandListCap ? s_list : nullptr;
    const bool near = kLong && len > kBandListCap && prunes_near(len, n_ops);
    const int m = len <= kBandListCap ? len : n_ops - first;
    constexpr int kPoints = kKind == 0 ? 1 : kStack ? 2 : 4;
    const int64_t base = (static_cast<int64_t>(s0[2]) * n[1] + s0[1]) * n[0] + s0[0];
    for (uint32_t q0 = static_cast<uint32_t>(wv) * 64 * kPoints; q0 < total;
         q0 += 64 * kPoints * W) {
      float p[kPoints][3], v[kPoints];
      int id[kPoints];
      uint64_t from = 0;
#pragma unroll
      for (int j = 0; j < kPoints; ++j) {
        const uint32_t q = q0 + 64 * j + lane;
        id[j] = s_queue[q < total ? q : total - 1];
        if (q0 + 64 * j < total) from |= s_from[(q0 >> 6) + j];
        const int blk = id[j] >> 6;
        p[j][0] = s_coord[1 + 4 * (blk & 3) + (id[j] & 3)];
        p[j][1] = s_coord[kBandCoords + 1 + (blk & 12) + ((id[j] >> 2) & 3)];
        p[j][2] = s_coord[2 * kBandCoords + 1 + 4 * (blk >> 4) + ((id[j] >> 4) & 3)];
      }
      // (spare points repeat the queue's last entry)
      from |= s_from[(total - 1) >> 6];
      if constexpr (kKind == 0)
        v[0] = sdf_eval_culled(C.ops, n_ops, p[0][0], p[0][1], p[0][2]);
      else if (near) {
        // (outside the leading scopes, which it enters itself)
#pragma unroll
        for (int j = 0; j < kPoints; ++j) {
          const int blk = id[j] >> 6;
          const int32_t at[3] = {s0[0] + 4 * (blk & 3) + (id[j] & 3),
                                 s0[1] + (blk & 12) + ((id[j] >> 2) & 3),
                                 s0[2] + 4 * (blk >> 4) + ((id[j] >> 4) & 3)};
#pragma unroll
          for (int a = 0; a < 3; ++a)
            p[j][a] = C.origin[a] + static_cast<float>(at[a]) * C.spacing[a];
        }
        sdf_eval_near<kPoints, kStack>(ops, n_ops, lane_ops(ops, 0, n_ops), p, v);
      } else
        sdf_eval_list<kPoints, kStack>(ops, first, list, s_mask, from, m, p, v);
#pragma unroll
      for (int j = 0; j < kPoints; ++j) {
        if (q0 + 64 * j + lane >= total) continue;
        const int blk = id[j] >> 6;
        const uint32_t x = 4 * (blk & 3) + (id[j] & 3), y = (blk & 12) + ((id[j] >> 2) & 3),
                       z = 4 * (blk >> 4) + ((id[j] >> 4) & 3);
        if (C.grid)
          (const_cast<float*>(C.grid) + base)[(z * static_cast<uint32_t>(n[1]) + y) *
                                                  static_cast<uint32_t>(n[0]) + x] = v[j];
        // classify_corners, distance.rs:52-54
        if (!(v[j] > 0.0f))
          atomicOr(reinterpret_cast<unsigned long long*>(&s_sign[blk]), 1ull << (id[j] & 63));
      }
    }
    __syncthreads();
    // Tiles add to kCounterLines lines in turn: thousands of them adding to
    // one word would wait for each other.
    if (threadIdx.x == 0) atomicAdd(evaluated + kCounterStride * (tile % kCounterLines), total);
  }
  store_tile_signs(C, s_sign, s0, tx, threadIdx.x, 64 * W);
}

// Cells whose marching-cubes case differs between two sign arrays of the
// same lattice (a band extraction's and the dense one's): a cell differs
// when any of its eight corner bits does.  One thread per 64-cell segment.
__global__ __launch_bounds__(256) void k_band_diff(Lattice L, McDims D, int64_t pitch_a,
                                                   const uint64_t* __restrict__ Sa,
                                                   const uint64_t* __restrict__ Sb,
                                                   unsigned long long* differing) {
  const int64_t nx = L.nx;
  const int64_t spr = D.segs_per_row;
  const int64_t cyn = L.ny - 1;
  uint32_t count = 0;
  for (int64_t g = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; g < D.n_segs;
       g += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    const int64_t row = g / spr, w = g - (g / spr) * spr;
    const int64_t cz = row / cyn, cy = row - (row / cyn) * cyn;
    uint64_t m = 0, n = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t row_k = (cz + (k >> 1)) * L.ny + cy + (k & 1);
      uint64_t na, nb;
      const uint64_t a = row_word(Sa, row_k * pitch_a + 64 * w, &na);
      const uint64_t b = row_word(Sb, row_k * nx + 64 * w, &nb);
      m |= a ^ b;
      n |= na ^ nb;
    }
    // cell i has corners at x = i and i + 1
    count += __popcll((m | (m >> 1) | (n << 63)) & seg_valid(nx, w));
  }
  unsigned long long c = count;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
  if (__lane_id() == 0 && c) atomicAdd(differing, c);
}

unsigned grid_of(uint64_t n, uint64_t cap) {
  uint64_t b = (n + 255) / 256;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return static_cast<unsigned>(b);
}

}  // namespace

BrickGrid brick_grid(const Lattice& L, int shift) {
  BrickGrid G;
  G.shift = shift;
  G.brick = 1 << shift;
  G.nbx = (L.nx - 1 + G.brick - 1) / G.brick;
  G.nby = (L.ny - 1 + G.brick - 1) / G.brick;
  G.nbz = (L.nz - 1 + G.brick - 1) / G.brick;
  G.n = G.nbx * G.nby * G.nbz;
  G.ncx = (G.nbx + kCoarse - 1) / kCoarse;
  G.ncy = (G.nby + kCoarse - 1) / kCoarse;
  G.ncz = (G.nbz + kCoarse - 1) / kCoarse;
  G.nc = G.ncx * G.ncy * G.ncz;
  return G;
}

hipError_t launch_coarse_certify(const DevOp* ops, int n_ops, const Lattice& L,
                                 const BrickGrid& G, uint8_t* coarse,
                                 unsigned long long* certified, hipStream_t s) {
  if (!ops || !coarse || !certified) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_coarse_certify, dim3(grid_of(G.nc, 1u << 30)), dim3(256), 0, s, ops, n_ops,
                     L, G, coarse, certified, certify_position_slack(L));
  return hipGetLastError();
}

hipError_t launch_brick_centres(const Lattice& L, const BrickGrid& G, float* centres,
                                float* half_diag, hipStream_t s) {
  hipLaunchKernelGGL(k_brick_centres, dim3(grid_of(G.n, 1u << 30)), dim3(256), 0, s, L, G,
                     centres, half_diag);
  return hipGetLastError();
}

float certify_position_slack(const Lattice& L) {
  // A lattice position origin + (float)i * spacing rounds twice (the
  // product and the sum), each by at most 2^-24 of the magnitude, so a
  // computed sample or centre coordinate is within 2^-23 M of the exact
  // lattice position, M bounding |origin| + i |spacing| over the lattice.
  // Two such points (centre and sample) add at most 2 sqrt(3) 2^-23 M to
  // their Euclidean distance.
  double m = 0.0;
  const int64_t n[3] = {L.nx, L.ny, L.nz};
  for (int a = 0; a < 3; ++a) {
    const double ma = std::fabs(static_cast<double>(L.origin[a])) +
                      static_cast<double>(n[a] > 0 ? n[a] - 1 : 0) *
                          std::fabs(static_cast<double>(L.spacing[a]));
    if (ma > m) m = ma;
  }
  return static_cast<float>(2.0 * std::sqrt(3.0) * std::ldexp(m, -23) * 1.01);
}

hipError_t launch_brick_certify(const DevOp* ops, int n_ops, const ProgramKind& kind,
                                const Lattice& L, const BrickGrid& G, const uint8_t* coarse,
                                const float* centres, const float* half_diag, uint8_t* proof,
                                unsigned long long* certified, hipStream_t s) {
  if (!ops || !coarse || !centres || !half_diag || !proof || !certified)
    return hipErrorInvalidValue;
  const uint64_t blocks = (static_cast<uint64_t>(G.nc) + 3) / 4;
  if (blocks > 0x7fffffffu) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  const float slack = certify_position_slack(L);
  if (!kind.bounded || !lattice_bounded(L)) {
    hipLaunchKernelGGL(k_brick_certify, grid, block, 0, s, ops, n_ops, G, coarse, centres,
                       half_diag, proof, certified, slack);
  } else {
    double m = kind.magnitude;
    const int64_t n[3] = {L.nx, L.ny, L.nz};
    for (int a = 0; a < 3; ++a)
      m = std::fmax(m, kind.magnitude + std::fabs(static_cast<double>(L.origin[a])) +
                           static_cast<double>(n[a]) * std::fabs(static_cast<double>(L.spacing[a])));
    const float mag = static_cast<float>(m * 1.001);
    if (kind.stack)
      hipLaunchKernelGGL(k_brick_certify_listed<true>, grid, block, 0, s, ops, n_ops, G, coarse,
                         centres, half_diag, proof, certified, slack, mag);
    else
      hipLaunchKernelGGL(k_brick_certify_listed<false>, grid, block, 0, s, ops, n_ops, G, coarse,
                         centres, half_diag, proof, certified, slack, mag);
  }
  return hipGetLastError();
}

hipError_t launch_brick_flags(const BrickGrid& G, const float* pred, const float* half_diag,
                              const uint8_t* proof, float margin, uint8_t* flags,
                              unsigned long long* n_band, unsigned long long* overturned,
                              hipStream_t s) {
  if ((!pred && !proof) || !flags || !n_band || !overturned) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_brick_flags, dim3(grid_of(static_cast<uint64_t>(G.n), 2048)), dim3(256), 0,
                     s, static_cast<uint64_t>(G.n), pred, half_diag, proof, margin, flags, n_band,
                     overturned);
  return hipGetLastError();
}

hipError_t launch_band_tiles(const DevOp* ops, int n_ops, const ProgramKind& kind,
                             const Lattice& L, const McDims& D, const BrickGrid& G,
                             const uint8_t* flags, const McBuffers& B, float* values,
                             unsigned long long* evaluated, hipStream_t s) {
  if (!ops || !flags || !B.signs || !evaluated || (D.sign_pitch & 63)) return hipErrorInvalidValue;
  const int64_t n_tiles = tile_count(L.nx, L.ny, L.nz);
  if (n_tiles > 0x7fffffff) return hipErrorInvalidValue;
  ResetArgs R;
  R.signs = B.signs;
  R.n_words = D.n_sign_words;
  R.agg = B.agg;
  R.incl = B.incl;
  R.n_blocks = D.n_blocks;
  R.totals = B.totals;
  const CellSpace C = single_cell_space(L, D, B.signs, ops, n_ops, values, nullptr);
  const bool few = n_tiles <= kBandFewTiles, more = n_ops > kBandListCap;
  const bool cull = !kind.bounded || !lattice_bounded(L) || (few && more);
  const auto culled = few ? k_band_tiles<0, kBandManyWaves, false> : k_band_tiles<0, kBandWaves, false>;
  const auto listed = more ? (kind.stack ? k_band_tiles<2, kBandWaves, true>
                                         : k_band_tiles<1, kBandWaves, true>)
                           : (kind.stack ? k_band_tiles<2, kBandWaves, false>
                                         : k_band_tiles<1, kBandWaves, false>);
  const auto kernel = cull ? culled : listed;
  const int waves = cull && few ? kBandManyWaves : kBandWaves;
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(n_tiles)),
                     dim3(static_cast<unsigned>(64 * waves)), 0, s, C, G, flags,
                     static_cast<uint32_t>(n_tiles), evaluated, R);
  return hipGetLastError();
}

hipError_t launch_band_diff(const Lattice& L, const McDims& D, int64_t pitch_a,
                            const uint64_t* signs_a,
                            const uint64_t* signs_b, unsigned long long* differing,
                            hipStream_t s) {
  if (!signs_a || !signs_b || !differing) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_band_diff, dim3(grid_of(static_cast<uint64_t>(D.n_segs), 16384)),
                     dim3(256), 0, s, L, D, pitch_a, signs_a, signs_b, differing);
  return hipGetLastError();
}

}  // namespace iso
