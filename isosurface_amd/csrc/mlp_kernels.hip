// Narrow-band network kernels for gfx950 (MI355X): MFMA forward, backward
// and Adam for the Fourier-feature MLP of mlp_kernels.h.
//
// MFMA tiling (v_mfma_f32_16x16x16_bf16, D = A B + C, 16x16 blocks):
//   A operand: lane l holds A[l % 16][4 (l / 16) + j], j = 0..3
//   B operand: lane l holds B[4 (l / 16) + j][l % 16]
//   D result:  lane l holds D[4 (l / 16) + j][l % 16]
// gfx950's double-K form (v_mfma_f32_16x16x32_bf16: lane l holds K values
// 8 (l / 16) + j, j = 0..7) takes two adjacent 16-wide K blocks at once: lane l
// passes its four values of block 2i then its four of block 2i+1, for A and B
// alike, which the instruction reads as one 32-wide block with its K index
// permuted the same way in both operands — the same sum of products.
// In each K block of features every lane evaluates the same function (sin or
// cos of one coordinate) at its own frequencies, c_k = 2^(k / 2) / 2 for
// k = 4 j + g, g = l / 16, i.e. c_g 4^j with c_g a power-of-two multiple of
// 1/2 or of sqrt(2)/2.
// A wavefront pushes 16 samples (the N dimension) through the network:
// layer outputs land in exactly the layout the next layer's B operand
// needs, so activations stay in registers from the features to the output.
// The backward-data pass uses the same layout with W^T fragments.  Weight
// gradients are products over the samples: the workgroup's 64 samples meet in
// LDS, unit by unit, which is the layout of both their operands.
#include <hip/hip_runtime.h>

#include "mlp_kernels.h"

namespace iso {
namespace mlp {

namespace {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4v __attribute__((ext_vector_type(4)));

// f32 -> bf16, nearest with ties to even (gfx950's v_cvt_pk_bf16_f32; a NaN
// stays a quiet NaN).
__device__ __forceinline__ uint16_t to_bf16(float f) {
  return __builtin_bit_cast(uint16_t, static_cast<__bf16>(f));
}

__device__ __forceinline__ float from_bf16(uint16_t b) {
  return __uint_as_float(static_cast<uint32_t>(b) << 16);
}

__device__ __forceinline__ f32x4 mfma(bf16x4 a, bf16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

// Two adjacent K blocks in one double-K MFMA (see the tiling note above).
__device__ __forceinline__ f32x4 mfma2(bf16x4 a0, bf16x4 a1, bf16x4 b0, bf16x4 b1, f32x4 c) {
  const s16x8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
  const s16x8 b = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Four f32 to bf16 (two v_cvt_pk_bf16_f32).
__device__ __forceinline__ bf16x4 pack4f(float a, float b, float c, float d) {
  return __builtin_bit_cast(bf16x4, __builtin_convertvector(f32x4v{a, b, c, d}, bf16x4v));
}

// Fragments of one 16-row block set, read from LDS: lane's 4 bf16 of block (mb, kb).
__device__ __forceinline__ bf16x4 frag(const uint16_t* F, int n_kb, int mb, int kb, int lane) {
  const uint16_t* p = F + ((mb * n_kb + kb) * 64 + lane) * 4;
  return *reinterpret_cast<const bf16x4*>(p);
}

// A lane's four features of K block kb for the point q (see the tiling note).
__device__ __forceinline__ bf16x4 features(const float* q, int kb, int lane) {
  const int g = lane >> 4;
  const float cg = __builtin_amdgcn_ldexpf((g & 1) ? 0x1.6a09e6p-1f : 0x1p-1f, g >> 1);
  float xf[4];
  if (kb < 6) {
    const float m = cg * q[kb % 3];  // c_k q for j = 0
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // c_g 4^j q: a power-of-two scaling of m, exact.  v_sin_f32 / v_cos_f32
      // take revolutions; the fraction of an f32 is exact, so reducing to it
      // changes nothing and keeps the argument in their input range.
      const float rev = __builtin_amdgcn_fractf(m * static_cast<float>(1 << (2 * j)));
      xf[j] = kb < 3 ? __builtin_amdgcn_sinf(rev) : __builtin_amdgcn_cosf(rev);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) xf[j] = g == 0 && j < 3 ? q[j] : 0.0f;
  }
  return pack4f(xf[0], xf[1], xf[2], xf[3]);
}

// Bias, ReLU and the bf16 rounding of a layer's 16 x 16 output block (b: the
// block's bias rows).
__device__ __forceinline__ bf16x4 activate(const f32x4& acc, const float* b, int r0) {
  return pack4f(fmaxf(acc[0] + b[r0 + 0], 0.0f), fmaxf(acc[1] + b[r0 + 1], 0.0f),
                fmaxf(acc[2] + b[r0 + 2], 0.0f), fmaxf(acc[3] + b[r0 + 3], 0.0f));
}

constexpr int kThreads = 256;
constexpr int kLdsFrags = kFragT2;  // forward fragments only (F1 F2 F3)

// Loads the first kN fragments and the bias block into LDS, with kT threads:
// every load is issued before the first is stored.
template <int kN, int kT>
__device__ __forceinline__ void load_model(const Model& M, uint16_t* sF, float* sB) {
  static_assert(kN % 8 == 0, "16-byte loads");
  constexpr int n = kN / 8, kRounds = (n + kT - 1) / kT;
  const uint4* src = reinterpret_cast<const uint4*>(M.frags);
  uint4* dst = reinterpret_cast<uint4*>(sF);
  const int t = static_cast<int>(threadIdx.x);
  uint4 v[kRounds];
#pragma unroll
  for (int i = 0; i < kRounds; ++i) {
    const int at = t + i * kT;
    v[i] = src[at < n ? at : 0];
  }
  // b1 b2 b3 w4 b4
  const int which = (t & 255) >> 6, k = t & 63;
  const int off = which == 0 ? kOffB1 : which == 1 ? kOffB2 : which == 2 ? kOffB3 : kOffW4;
  static_assert(kHidden == 64 && kT >= 4 * kHidden, "one bias a thread");
  const float bias = M.theta[off + k], last = M.theta[kOffB4];
#pragma unroll
  for (int i = 0; i < kRounds; ++i) {
    const int at = t + i * kT;
    if (at < n) dst[at] = v[i];
  }
  if (t < 4 * kHidden) sB[t] = bias;
  if (t == 0) sB[4 * kHidden] = last;
}

// Inference forward of kT 16-sample tiles at once: every weight fragment
// read from LDS feeds all kT tiles' MFMAs, 1/kT of the LDS traffic per
// sample of one tile at a time.  Pairs of K blocks go through double-K
// MFMAs.  p[t]: this lane's sample of tile t (lane l's sample is l % 16);
// f[t]: its output.
template <int kT>
__device__ __forceinline__ void forward_tiles(const uint16_t* sF, const float* sB,
                                              const float (*p)[3], int lane, float* f) {
  const int r0 = 4 * (lane >> 4);
  const uint16_t* F1 = sF + kFragF1;
  const uint16_t* F2 = sF + kFragF2;
  const uint16_t* F3 = sF + kFragF3;
  const float* b1 = sB;
  const float* b2 = sB + kHidden;
  const float* b3 = sB + 2 * kHidden;
  const float* w4 = sB + 3 * kHidden;
  const float b4 = sB[4 * kHidden];
  f32x4 z[kT][4];
#pragma unroll
  for (int t = 0; t < kT; ++t)
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) z[t][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
  for (int kb = 0; kb + 1 < kKB1; kb += 2) {
    bf16x4 x0[kT], x1[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) {
      x0[t] = features(p[t], kb, lane);
      x1[t] = features(p[t], kb + 1, lane);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const bf16x4 w0 = frag(F1, kKB1, mb, kb, lane), w1 = frag(F1, kKB1, mb, kb + 1, lane);
#pragma unroll
      for (int t = 0; t < kT; ++t) z[t][mb] = mfma2(w0, w1, x0[t], x1[t], z[t][mb]);
    }
  }
  if (kKB1 & 1) {
    bf16x4 x[kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) x[t] = features(p[t], kKB1 - 1, lane);
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const bf16x4 w = frag(F1, kKB1, mb, kKB1 - 1, lane);
#pragma unroll
      for (int t = 0; t < kT; ++t) z[t][mb] = mfma(w, x[t], z[t][mb]);
    }
  }
  bf16x4 h[kT][4];
#pragma unroll
  for (int t = 0; t < kT; ++t)
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) h[t][mb] = activate(z[t][mb], b1 + 16 * mb, r0);
  // Hidden layers 2 and 3 (W2, W3): 64-wide K, two double-K MFMAs a block.
  auto layer = [&](const uint16_t* F, const float* b) {
    bf16x4 y[kT][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      f32x4 a[kT];
#pragma unroll
      for (int t = 0; t < kT; ++t) a[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kp = 0; kp < 4; kp += 2) {
        const bf16x4 w0 = frag(F, 4, mb, kp, lane), w1 = frag(F, 4, mb, kp + 1, lane);
#pragma unroll
        for (int t = 0; t < kT; ++t) a[t] = mfma2(w0, w1, h[t][kp], h[t][kp + 1], a[t]);
      }
#pragma unroll
      for (int t = 0; t < kT; ++t) y[t][mb] = activate(a[t], b + 16 * mb, r0);
    }
#pragma unroll
    for (int t = 0; t < kT; ++t)
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) h[t][mb] = y[t][mb];
  };
  layer(F2, b2);
  layer(F3, b3);
#pragma unroll
  for (int t = 0; t < kT; ++t) {
    float q = 0.0f;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        q += w4[16 * mb + r0 + j] * from_bf16(static_cast<uint16_t>(h[t][mb][j]));
    // The four lanes of a sample (l, l^16, l^32, l^48) hold its 64 terms.
    q += __shfl_xor(q, 16, 64);
    q += __shfl_xor(q, 32, 64);
    f[t] = q + b4;
  }
}

// Tiles of 16 samples per fragment read in the inference forward.
constexpr int kFwdTiles = 4;
// 512 threads: the fragments' 40 KB of LDS then allow as many waves per SIMD
// as the registers do.
constexpr int kFwdThreads = 512;

__global__ __launch_bounds__(kFwdThreads) void k_forward(Model M, const float* __restrict__ points,
                                                         int64_t n, float* __restrict__ out) {
  __shared__ __align__(16) uint16_t sF[kLdsFrags];
  __shared__ float sB[4 * kHidden + 1];
  load_model<kLdsFrags, kFwdThreads>(M, sF, sB);
  __syncthreads();
  const int lane = __lane_id();
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kFwdThreads / 64) + (threadIdx.x >> 6);
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * (kFwdThreads / 64);
  constexpr int64_t kStep = 16 * kFwdTiles;
  for (int64_t t0 = wave * kStep; t0 < n; t0 += n_waves * kStep) {
    // The fragments are re-read from LDS for every kFwdTiles tiles rather
    // than held in registers across them: fewer registers, more waves per
    // SIMD.
    asm volatile("" ::: "memory");
    float p[kFwdTiles][3], f[kFwdTiles];
#pragma unroll
    for (int t = 0; t < kFwdTiles; ++t) {
      const int64_t si = t0 + 16 * t + (lane & 15);
#pragma unroll
      for (int a = 0; a < 3; ++a) p[t][a] = si < n ? points[3 * si + a] : 0.0f;
    }
    forward_tiles<kFwdTiles>(sF, sB, p, lane, f);
    if (lane < 16) {
#pragma unroll
      for (int t = 0; t < kFwdTiles; ++t) {
        const int64_t si = t0 + 16 * t + lane;
        if (si < n) out[si] = f[t];
      }
    }
  }
}

__device__ __forceinline__ uint32_t hash32(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t h = a * 0x9E3779B1u ^ (b + 0x85EBCA77u) * 0xC2B2AE3Du ^ (c + 0x27D4EB2Fu) * 0x165667B1u;
  h ^= h >> 15;
  h *= 0x2C1B3C6Du;
  h ^= h >> 12;
  h *= 0x297A2D39u;
  h ^= h >> 15;
  return h;
}

// Forward and backward of one batch.  A workgroup takes kGroup samples at a
// time: each of its four wavefronts runs 16 of them forward and back through
// the data path in registers, leaving the bf16 activations and their
// derivatives in LDS, unit by unit; then wavefront w multiplies rows 16w..16w+15
// of every layer's derivatives with the layer's inputs over the 64 samples
// (15 blocks of 16 x 16, accumulated in registers over the workgroup's
// groups).  Its gradient goes to a row of its own: no atomics, and the same
// sums on every run.  Bound by the latency of one wavefront's chain on each
// SIMD (a batch of 16384 is one group a CU): 21 us a step with the Adam
// kernel, where activations through memory, their re-reading by one wavefront
// per block and f32 atomics took 73 us.
constexpr int kPitch = kGroup + 8;  // samples of an LDS row: 16-byte rows, spread over the banks
constexpr int kRowX = 0, kRowH1 = kRowX + kFeatPad, kRowH2 = kRowH1 + kHidden,
              kRowH3 = kRowH2 + kHidden, kRowD1 = kRowH3 + kHidden, kRowD2 = kRowD1 + kHidden,
              kRowD3 = kRowD2 + kHidden, kLdsRows = kRowD3 + kHidden;

__global__ __launch_bounds__(kThreads) void k_train(Model M, Batch B, Samples S, uint32_t step) {
  __shared__ __align__(16) uint16_t sF[kFrags];
  __shared__ __align__(16) uint16_t sA[kLdsRows * kPitch];
  __shared__ float sB[4 * kHidden + 1];
  __shared__ float sG[kGroup];
  __shared__ float sSum[2][kThreads / 64];
  load_model<kFrags, kThreads>(M, sF, sB);
  const int lane = __lane_id();
  const int wv = static_cast<int>(threadIdx.x >> 6);
  const int r0 = 4 * (lane >> 4);
  const int col = lane & 15;
  const float* w4 = sB + 3 * kHidden;
  const float inv_n = 1.0f / static_cast<float>(B.n);
  const int64_t n_groups = (B.n + kGroup - 1) / kGroup;
  // rows first + 4 (lane / 16) + j of an LDS block, this wavefront's sample col
  auto keep = [&](int first, const bf16x4& v) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      sA[(first + r0 + j) * kPitch + 16 * wv + col] = static_cast<uint16_t>(v[j]);
  };
  f32x4 acc1[kKB1], acc2[4], acc3[4];  // rows 16 wv of dW1, dW2, dW3
#pragma unroll
  for (int i = 0; i < kKB1; ++i) acc1[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < 4; ++i) acc2[i] = acc3[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float unit_sum = 0.0f;             // this thread's bias or output weight
  float loss = 0.0f, g_sum = 0.0f;  // lanes 0..15
  for (int64_t grp = blockIdx.x; grp < n_groups; grp += gridDim.x) {
    __syncthreads();  // the fragments are there; the last group's rows are read
    const int64_t s = grp * kGroup + 16 * wv + col;
    const bool live = s < B.n;  // (the same for a whole wavefront)
    float q[3] = {0.0f, 0.0f, 0.0f}, t = 0.0f, wgt = 0.0f;
    if (live) {
      uint64_t src = static_cast<uint64_t>(s);
      if (S.gather) {
        const uint32_t h = hash32(S.seed, step, static_cast<uint32_t>(s));
        src = S.count > 0xffffffffull ? h : h % static_cast<uint32_t>(S.count);
      }
      q[0] = S.points[3 * src];
      q[1] = S.points[3 * src + 1];
      q[2] = S.points[3 * src + 2];
      t = fminf(fmaxf(S.sdf[src], -S.clamp), S.clamp);
      wgt = S.weight ? S.weight[src] : 1.0f;
    }
    // forward
    bf16x4 h1[4], h2[4], h3[4];
    {
      f32x4 z[4];
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) z[mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kb = 0; kb + 1 < kKB1; kb += 2) {
        const bf16x4 x0 = features(q, kb, lane), x1 = features(q, kb + 1, lane);
        keep(kRowX + 16 * kb, x0);
        keep(kRowX + 16 * kb + 16, x1);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
          z[mb] = mfma2(frag(sF + kFragF1, kKB1, mb, kb, lane),
                        frag(sF + kFragF1, kKB1, mb, kb + 1, lane), x0, x1, z[mb]);
      }
      static_assert(kKB1 & 1, "the last feature block stands alone");
      const bf16x4 x = features(q, kKB1 - 1, lane);
      keep(kRowX + 16 * (kKB1 - 1), x);
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) {
        z[mb] = mfma(frag(sF + kFragF1, kKB1, mb, kKB1 - 1, lane), x, z[mb]);
        h1[mb] = activate(z[mb], sB + 16 * mb, r0);
        keep(kRowH1 + 16 * mb, h1[mb]);
      }
    }
    // A 64-wide K product with fragment set F.
    auto product64 = [&](const uint16_t* F, int mb, const bf16x4* h) {
      f32x4 a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kp = 0; kp < 4; kp += 2)
        a = mfma2(frag(F, 4, mb, kp, lane), frag(F, 4, mb, kp + 1, lane), h[kp], h[kp + 1], a);
      return a;
    };
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      h2[mb] = activate(product64(sF + kFragF2, mb, h1), sB + kHidden + 16 * mb, r0);
      keep(kRowH2 + 16 * mb, h2[mb]);
    }
    float f = 0.0f;
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      h3[mb] = activate(product64(sF + kFragF3, mb, h2), sB + 2 * kHidden + 16 * mb, r0);
      keep(kRowH3 + 16 * mb, h3[mb]);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        f += w4[16 * mb + r0 + j] * from_bf16(static_cast<uint16_t>(h3[mb][j]));
    }
    // The four lanes of a sample (l, l^16, l^32, l^48) hold its 64 terms.
    f += __shfl_xor(f, 16, 64);
    f += __shfl_xor(f, 32, 64);
    f += sB[4 * kHidden];
    // Least squares plus (overshoot - 1) e^2, e the part of the error that
    // lies outside the interval between 0 and the target.
    const float r = f - t;
    const float e = f - fminf(fmaxf(f, fminf(t, 0.0f)), fmaxf(t, 0.0f));
    const float ow = S.overshoot - 1.0f;
    const float g = live ? wgt * (r + ow * e) * inv_n : 0.0f;
    if (lane < 16) {
      if (live) loss += wgt * (r * r + ow * e * e);
      g_sum += g;
      sG[16 * wv + col] = g;
    }
    // dz3 = bf16(g w4 [h3 > 0]), dz2 = bf16((W3^T dz3) [h2 > 0]), dz1 likewise.
    auto gate = [&](const f32x4& a, const bf16x4& h) {
      float d[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
        d[j] = from_bf16(static_cast<uint16_t>(h[j])) > 0.0f ? a[j] : 0.0f;
      return pack4f(d[0], d[1], d[2], d[3]);
    };
    bf16x4 d3[4], d2[4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      f32x4 a;
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = g * w4[16 * mb + r0 + j];
      d3[mb] = gate(a, h3[mb]);
      keep(kRowD3 + 16 * mb, d3[mb]);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      d2[mb] = gate(product64(sF + kFragT3, mb, d3), h2[mb]);
      keep(kRowD2 + 16 * mb, d2[mb]);
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
      keep(kRowD1 + 16 * mb, gate(product64(sF + kFragT2, mb, d2), h1[mb]));
    __syncthreads();

    // Weight gradients: block rows 16 wv, K = the 64 samples in two halves; lane
    // l holds row l % 16 at samples 32 half + 8 (l / 16) .. + 7 of either operand.
    auto operand = [&](int row, int half) {
      return *reinterpret_cast<const bf16x8*>(sA + (row + col) * kPitch + 32 * half +
                                              8 * (lane >> 4));
    };
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const bf16x8 a1 = operand(kRowD1 + 16 * wv, half), a2 = operand(kRowD2 + 16 * wv, half),
                   a3 = operand(kRowD3 + 16 * wv, half);
#pragma unroll
      for (int nb = 0; nb < kKB1; ++nb)
        acc1[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, operand(kRowX + 16 * nb, half),
                                                           acc1[nb], 0, 0, 0);
#pragma unroll
      for (int nb = 0; nb < 4; ++nb) {
        acc2[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, operand(kRowH1 + 16 * nb, half),
                                                           acc2[nb], 0, 0, 0);
        acc3[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a3, operand(kRowH2 + 16 * nb, half),
                                                           acc3[nb], 0, 0, 0);
      }
    }
    // Thread i: db of unit i (threads 0-191: dz1, dz2, dz3) or dw4 of unit i - 192.
    {
      const int i = static_cast<int>(threadIdx.x);
      const uint16_t* row = sA + (i < 192 ? kRowD1 + i : kRowH3 + i - 192) * kPitch;
#pragma unroll
      for (int k = 0; k < kGroup; k += 8) {
        const s16x8 v = *reinterpret_cast<const s16x8*>(row + k);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = from_bf16(static_cast<uint16_t>(v[j]));
          unit_sum += i < 192 ? x : sG[k + j] * x;
        }
      }
    }
  }
  // The workgroup's row: W1's columns stay in the kernels' feature order.
  float* row = B.rows + static_cast<int64_t>(blockIdx.x) * kGradRow;
  auto store = [&](int off, int cols, int nb, const f32x4& a) {
#pragma unroll
    for (int j = 0; j < 4; ++j) row[off + (16 * wv + r0 + j) * cols + 16 * nb + col] = a[j];
  };
#pragma unroll
  for (int nb = 0; nb < kKB1; ++nb) store(kOffW1, kFeatPad, nb, acc1[nb]);
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    store(kOffW2, kHidden, nb, acc2[nb]);
    store(kOffW3, kHidden, nb, acc3[nb]);
  }
  {
    const int i = static_cast<int>(threadIdx.x);
    const int off = i < 64 ? kOffB1 : i < 128 ? kOffB2 : i < 192 ? kOffB3 : kOffW4;
    row[off + (i & 63)] = unit_sum;
  }
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) {
    loss += __shfl_xor(loss, d, 64);
    g_sum += __shfl_xor(g_sum, d, 64);
  }
  if (lane == 0) {
    sSum[0][wv] = g_sum;
    sSum[1][wv] = loss;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    row[kOffB4] = (sSum[0][0] + sSum[0][1]) + (sSum[0][2] + sSum[0][3]);
    row[kParams] = (sSum[1][0] + sSum[1][1]) + (sSum[1][2] + sSum[1][3]);
  }
}

// Feature row in the kernels' order of feature column c of the parameters,
// and the reverse.
__device__ __forceinline__ int feature_row(int c) {
  if (c < 3) return 96 + c;       // coordinates
  if (c >= kFeat) return c;       // padding
  const int q = c - 3, k = q / 6, t = q - 6 * k;  // frequency k, function t
  return 16 * t + 4 * (k & 3) + (k >> 2);
}
__device__ __forceinline__ int feature_column(int r) {
  if (r >= kFeat) return r;
  if (r >= 96) return r - 96;
  const int t = r >> 4, i = r & 15;
  return 3 + 6 * ((i >> 2) + 4 * (i & 3)) + t;
}

// Fragment slot of parameter p (weights of layers 1-3), and of its transpose
// (layers 2-3).
__device__ __forceinline__ void frag_slots(int p, int* f, int* ft) {
  *f = -1;
  *ft = -1;
  int base, cols, kbn, fbase, tbase;
  if (p < kOffB1) {
    base = kOffW1, cols = kFeatPad, kbn = kKB1, fbase = kFragF1, tbase = -1;
  } else if (p >= kOffW2 && p < kOffB2) {
    base = kOffW2, cols = kHidden, kbn = 4, fbase = kFragF2, tbase = kFragT2;
  } else if (p >= kOffW3 && p < kOffB3) {
    base = kOffW3, cols = kHidden, kbn = 4, fbase = kFragF3, tbase = kFragT3;
  } else {
    return;
  }
  const int q = p - base;
  const int row = q / cols;
  int c = q - row * cols;
  if (base == kOffW1) c = feature_row(c);
  // W[row][c] sits in block (row / 16, c / 16) at lane (row % 16) + 16 ((c % 16) / 4), slot c % 4
  *f = fbase + (((row >> 4) * kbn + (c >> 4)) * 64 + (row & 15) + 16 * ((c & 15) >> 2)) * 4 + (c & 3);
  if (tbase >= 0) {
    // W^T[c][row]: block (c / 16, row / 16), lane (c % 16) + 16 ((row % 16) / 4), slot row % 4
    *ft = tbase + (((c >> 4) * 4 + (row >> 4)) * 64 + (c & 15) + 16 * ((row & 15) >> 2)) * 4 +
          (row & 3);
  }
}

__global__ __launch_bounds__(kThreads) void k_pack(Model M) {
  const int p = blockIdx.x * kThreads + threadIdx.x;
  if (p >= kParams) return;
  int f, ft;
  frag_slots(p, &f, &ft);
  const uint16_t b = to_bf16(M.theta[p]);
  if (f >= 0) M.frags[f] = b;
  if (ft >= 0) M.frags[ft] = b;
}

// The sum of the batch's rows, and with kStep the Adam step from it.  A
// workgroup takes 32 neighbouring entries; 32 threads read a row's 128 bytes
// of them and the 8 sets of threads every eighth row, so the chip reads the
// 16 MB of a full batch's rows at once.
constexpr int kSumSlots = 32, kSumParts = kThreads / kSumSlots;

template <bool kStep>
__global__ __launch_bounds__(kThreads) void k_adam(Model M, const float* __restrict__ rows,
                                                   int n_rows, float lr, float beta1, float beta2,
                                                   float eps, float c1, float c2) {
  __shared__ float s_part[kSumParts][kSumSlots];
  const int i = static_cast<int>(threadIdx.x) % kSumSlots, part = threadIdx.x / kSumSlots;
  const int slot = blockIdx.x * kSumSlots + i;
  float sum = 0.0f;
  if (slot <= kParams) {
#pragma unroll 8
    for (int r = part; r < n_rows; r += kSumParts)
      sum += rows[static_cast<int64_t>(r) * kGradRow + slot];
  }
  s_part[part][i] = sum;
  __syncthreads();
  if (part != 0 || slot > kParams) return;
#pragma unroll
  for (int k = 1; k < kSumParts; ++k) sum += s_part[k][i];
  if (slot == kParams) {
    M.loss[0] = sum;
    return;
  }
  int p = slot;
  if (slot < kOffB1) {
    const int row = slot / kFeatPad;
    p = row * kFeatPad + feature_column(slot - row * kFeatPad);
  }
  if (!kStep) {
    M.grad[p] = sum;
    return;
  }
  const float g = sum;
  const float m = beta1 * M.m[p] + (1.0f - beta1) * g;
  const float v = beta2 * M.v[p] + (1.0f - beta2) * g * g;
  M.m[p] = m;
  M.v[p] = v;
  const float w = M.theta[p] - lr * (m / c1) / (sqrtf(v / c2) + eps);
  M.theta[p] = w;
  int f, ft;
  frag_slots(p, &f, &ft);
  const uint16_t b = to_bf16(w);
  if (f >= 0) M.frags[f] = b;
  if (ft >= 0) M.frags[ft] = b;
}

unsigned blocks_for(int64_t n) { return static_cast<unsigned>((n + kThreads - 1) / kThreads); }

}  // namespace

hipError_t launch_pack(const Model& M, hipStream_t s) {
  hipLaunchKernelGGL(k_pack, dim3(blocks_for(kParams)), dim3(kThreads), 0, s, M);
  return hipGetLastError();
}

hipError_t launch_forward(const Model& M, const float* points, int64_t n, float* out,
                          hipStream_t s) {
  if (n <= 0) return hipSuccess;
  constexpr int64_t per_block = 16 * kFwdTiles * (kFwdThreads / 64);  // kFwdTiles tiles per wavefront
  int64_t blocks = (n + per_block - 1) / per_block;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_forward, dim3(static_cast<unsigned>(blocks)), dim3(kFwdThreads), 0, s, M,
                     points, n, out);
  return hipGetLastError();
}

hipError_t launch_train_batch(const Model& M, const Batch& B, const Samples& S, uint32_t step,
                              hipStream_t s) {
  if (B.n <= 0 || (B.n & 15) || S.count == 0 || !B.rows) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_train, dim3(static_cast<unsigned>(batch_rows(B.n))), dim3(kThreads), 0, s, M,
                     B, S, step);
  return hipGetLastError();
}

namespace {
constexpr unsigned kSumBlocks = (kParams + 1 + kSumSlots - 1) / kSumSlots;
}

hipError_t launch_adam(const Model& M, const Batch& B, uint32_t step, float lr, float beta1,
                       float beta2, float eps, hipStream_t s) {
  const double c1 = 1.0 - __builtin_pow(static_cast<double>(beta1), static_cast<double>(step));
  const double c2 = 1.0 - __builtin_pow(static_cast<double>(beta2), static_cast<double>(step));
  hipLaunchKernelGGL(k_adam<true>, dim3(kSumBlocks), dim3(kThreads), 0, s, M, B.rows,
                     batch_rows(B.n), lr, beta1, beta2, eps, static_cast<float>(c1),
                     static_cast<float>(c2));
  return hipGetLastError();
}

hipError_t launch_gradient(const Model& M, const Batch& B, hipStream_t s) {
  hipLaunchKernelGGL(k_adam<false>, dim3(kSumBlocks), dim3(kThreads), 0, s, M, B.rows,
                     batch_rows(B.n), 0.0f, 0.0f, 0.0f, 0.0f, 1.0f, 1.0f);
  return hipGetLastError();
}

}  // namespace mlp
}  // namespace iso
