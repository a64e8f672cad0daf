// Interval evaluation and list evaluation of lowered SDF programs for a
// wavefront that works on one tile of a lattice (see sparse_kernels.hip).
//
// Intervals: every operation of a program's f32 evaluation is monotone in
// each |coordinate difference| or operand (a correctly rounded operation is
// monotone because the exact one is), so evaluating the same operations at
// the least and the greatest |q_c| of a box gives bounds that no f32
// evaluation at a point of the box leaves.  Two operations take an allowance:
// square roots, which the bounds take from the hardware's approximation, and
// the polynomial smooth minimum, monotone only in exact arithmetic.
//
// The bounds hold for finite parameters and coordinates of ordinary
// magnitude (no overflow of a square): the host checks that (program_bounded
// and lattice_bounded, sparse_kernels.h), and programs or lattices beyond it
// are evaluated densely.
//
// kStack: the program holds values below the running one (a push after the
// first).  Most programs do not, and the interpreters without a stack carry a
// third of the state through their branches.
#pragma once
#include <hip/hip_runtime.h>

#include "mc_kernels.h"
#include "sdf_eval.h"
#include "sdf_program.h"

namespace iso {

// Bounds of the correctly rounded square root by the hardware's, which is
// within one ulp of it (two for certain: four are allowed), and within 2^-62
// of it where its operand is too small to be normal.
__device__ __forceinline__ float sqrt_below(float x) {
  return __builtin_amdgcn_sqrtf(x) * 0.99999976f;  // 1 - 2^-22
}
__device__ __forceinline__ float sqrt_above(float x) {
  return __builtin_fmaf(__builtin_amdgcn_sqrtf(x), 1.00000024f, 1.0e-18f);  // 1 + 2^-22
}

// Bounds of a primitive's f32 value over the points of the box [lo, hi]
// (after the primitive's own translation).
__device__ __forceinline__ void prim_interval(uint32_t code, const float* prm, const float* lo,
                                              const float* hi, float* vlo, float* vhi) {
  float an[3], af[3];  // least and greatest |q_c|
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    an[a] = fmaxf(fmaxf(lo[a], -hi[a]), 0.0f);
    af[a] = fmaxf(-lo[a], hi[a]);
  }
  // All but the torus are nondecreasing in each |q_c|.
  if (code == kSphere) {
    *vlo = sqrt_below((an[0] * an[0] + an[1] * an[1]) + an[2] * an[2]) - prm[0];
    *vhi = sqrt_above((af[0] * af[0] + af[1] * af[1]) + af[2] * af[2]) - prm[0];
  } else if (code == kBox) {
    float n[3], f[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      an[a] = an[a] - prm[a];
      af[a] = af[a] - prm[a];
      n[a] = fmaxf(an[a], 0.0f);
      f[a] = fmaxf(af[a], 0.0f);
    }
    *vlo = sqrt_below((n[0] * n[0] + n[1] * n[1]) + n[2] * n[2]) +
           fminf(fmaxf(an[0], fmaxf(an[1], an[2])), 0.0f);
    *vhi = sqrt_above((f[0] * f[0] + f[1] * f[1]) + f[2] * f[2]) +
           fminf(fmaxf(af[0], fmaxf(af[1], af[2])), 0.0f);
  } else {
    // distance to the axis circle or surface
    const float q0 = sqrt_below(an[0] * an[0] + an[1] * an[1]) - prm[0];
    const float q1 = sqrt_above(af[0] * af[0] + af[1] * af[1]) - prm[0];
    if (code == kTorus) {  // nondecreasing in |q| and |z|
      const float qn = fmaxf(fmaxf(q0, -q1), 0.0f), qf = fmaxf(-q0, q1);
      *vlo = sqrt_below(qn * qn + an[2] * an[2]) - prm[1];
      *vhi = sqrt_above(qf * qf + af[2] * af[2]) - prm[1];
    } else {  // kCylinder
      const float z0 = an[2] - prm[1], z1 = af[2] - prm[1];
      const float dx0 = fmaxf(q0, 0.0f), dz0 = fmaxf(z0, 0.0f);
      const float dx1 = fmaxf(q1, 0.0f), dz1 = fmaxf(z1, 0.0f);
      *vlo = fminf(fmaxf(q0, z0), 0.0f) + sqrt_below(dx0 * dx0 + dz0 * dz0);
      *vhi = fminf(fmaxf(q1, z1), 0.0f) + sqrt_above(dx1 * dx1 + dz1 * dz1);
    }
  }
}

// Wave-wide minima by data-parallel primitives: a register move each, where a
// shuffle goes through the LDS unit and takes about a hundred cycles.
constexpr float kNoBound = 3.0e38f;

template <int kCtrl, int kRows>
__device__ __forceinline__ float dpp_min(float v) {
  const int t = __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, kNoBound),
                                            __builtin_bit_cast(int, v), kCtrl, kRows, 0xf, false);
  return fminf(v, __builtin_bit_cast(float, t));
}
// Inclusive prefix minimum over the lanes (values at most kNoBound).
__device__ __forceinline__ float wave_min_upto(float v) {
  v = dpp_min<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8: within rows of 16 lanes
  v = dpp_min<0x112, 0xf>(v);
  v = dpp_min<0x114, 0xf>(v);
  v = dpp_min<0x118, 0xf>(v);
  v = dpp_min<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_min<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
// The minimum over all lanes, in every lane.
__device__ __forceinline__ float wave_min(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wave_min_upto(v)), 63));
}
// The minimum over the lanes below this one.
__device__ __forceinline__ float wave_min_before(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, kNoBound),
                                         __builtin_bit_cast(int, wave_min_upto(v)), 0x138, 0xf, 0xf,
                                         false));  // wave_shr:1
}

// Whether an operand of a smooth minimum that is at least `gap` above the
// running value leaves it unchanged (the blend weight is then exactly 0).
__device__ __forceinline__ bool smooth_inactive(float gap, float k) {
  constexpr float u = 5.9604645e-08f;  // 2^-24
  return gap * (1.0f - 4.0f * u) >= k * (1.0f + 4.0f * u);
}

// Bounds of smooth_min over operands in [alo, ahi] and [blo, bhi].
__device__ __forceinline__ void smooth_interval(float alo, float ahi, float blo, float bhi, float k,
                                                float* lo, float* hi) {
  constexpr float u = 5.9604645e-08f;
  const float mag = fmaxf(fmaxf(__builtin_fabsf(alo), __builtin_fabsf(ahi)),
                          fmaxf(__builtin_fabsf(blo), __builtin_fabsf(bhi)));
  const float slack = 32.0f * u * (k + mag);
  *lo = smooth_min(alo, blo, k) - slack;
  *hi = smooth_min(ahi, bhi, k) + slack;
}

// The running bounds of a program's evaluation.
template <bool kStack>
struct Bounds {
  // Before the first value: neutral to min, as the first push is read.
  float lo = kNoBound, hi = kNoBound;
  bool have_top = false;
  ShiftStack slo, shi;
  __device__ __forceinline__ Bounds() {
#pragma unroll
    for (int i = 0; i < kMaxValueStack; ++i) slo.v[i] = shi.v[i] = 0.0f;
  }
  // Joins a primitive bounded by [vlo, vhi]; returns false, with the bounds as
  // they were, when for every lane with `active` the operand leaves the
  // running value bit for bit as it is at every point of the lane's box:
  //   min:         its lower bound exceeds the running upper bound,
  //   smooth min:  it does by the blend width (the weight is then exactly 0),
  //   max, max of the negated operand: its upper bound is below the running
  //                lower bound.
  // *matters: the lanes for which it does not.
  __device__ __forceinline__ bool join(uint32_t mode, float k, float vlo, float vhi, bool active,
                                       uint64_t* matters) {
    if (kStack && mode == kPush) {
      if (have_top) {
        slo.push(lo);
        shi.push(hi);
      }
      have_top = true;
      lo = vlo;
      hi = vhi;
      *matters = ~0ull;
      return true;
    }
    bool idle;
    float nlo, nhi;
    if (mode == kMin || (!kStack && mode == kPush)) {
      idle = vlo > hi;
      nlo = fminf(lo, vlo);
      nhi = fminf(hi, vhi);
    } else if (mode == kSmooth) {
      idle = smooth_inactive(vlo - hi, k);
      smooth_interval(lo, hi, vlo, vhi, k, &nlo, &nhi);
    } else {
      // max(top, v), max(v, -top) or max(top, -v)
      const float al = mode == kDiff ? -hi : lo, ah = mode == kDiff ? -lo : hi;
      const float bl = mode == kDiffRev ? -vhi : vlo, bh = mode == kDiffRev ? -vlo : vhi;
      idle = mode != kDiff && bh < al;
      nlo = fmaxf(al, bl);
      nhi = fmaxf(ah, bh);
    }
    *matters = __ballot(active && !idle);
    if (*matters == 0ull) return false;
    lo = nlo;
    hi = nhi;
    return true;
  }
  // A binary operator on (below, top).
  __device__ __forceinline__ void operate(uint32_t code, float k) {
    const float tl = lo, th = hi;
    const float wl = slo.pop(), wh = shi.pop();
    if (code == kUnion) {
      lo = fminf(wl, tl);
      hi = fminf(wh, th);
    } else if (code == kSmoothUnion) {
      smooth_interval(wl, wh, tl, th, k, &lo, &hi);
    } else {
      // max(w, t), max(t, -w) or max(w, -t)
      const bool nw = code == kDifference, nt = code == kDifferenceRev;
      lo = fmaxf(nw ? -wh : wl, nt ? -th : tl);
      hi = fmaxf(nw ? -wl : wh, nt ? -tl : th);
    }
  }
};

// Moves a box into or out of a translation scope: [cl, ch] is the base box
// [bl, bh] less the offsets of the open scopes, outermost first.
__device__ __forceinline__ void enter_scope(OpsPtr ops, int op, float* cl, float* ch) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    cl[a] = cl[a] - ops[op].off[a];
    ch[a] = ch[a] - ops[op].off[a];
  }
}
__device__ __forceinline__ void restore_scopes(OpsPtr ops, const ScopeStack& scopes,
                                               const float* bl, const float* bh, float* cl,
                                               float* ch) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    cl[a] = bl[a];
    ch[a] = bh[a];
  }
  for (int s = 0; s < scopes.depth; ++s) enter_scope(ops, scopes.at(s), cl, ch);
}

__device__ __forceinline__ void op_interval(const DevOp& op, const float* cl, const float* ch,
                                            float* vlo, float* vhi) {
  float ql[3], qh[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {  // (an untranslated primitive's offset is 0, and x - 0 is x)
    ql[a] = cl[a] - op.off[a];
    qh[a] = ch[a] - op.off[a];
  }
  prim_interval(op.code, op.prm, ql, qh, vlo, vhi);
}

// The same for a primitive's Directed value, three components of which each is
// the signed distance along its axis, or kDirectedMiss where the axis' line
// misses the shape.  They are ordered by what is known of all three:
//   4         all kDirectedMiss at every point of the box: no component of any
//             other value is greater;
//   1 to 3    all positive; -1 to -3: all negative; -3 to 3: not known.
// (The negatives' bounds mirror these.)  Minima and maxima of values follow
// those of the bounds, so Bounds combines them, and what it finds idle leaves
// every component as it is.  A torus is not bounded.
__device__ __forceinline__ void directed_interval(const DevOp& op, const float* cl,
                                                  const float* ch, float* vlo, float* vhi) {
  float an[3], af[3];  // least and greatest |q_c|
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float lo = cl[a] - op.off[a], hi = ch[a] - op.off[a];
    an[a] = fmaxf(fmaxf(lo, -hi), 0.0f);
    af[a] = fmaxf(-lo, hi);
  }
  bool out[3];        // outside along the axis
  bool in = true;     // all negative
  if (op.code == kBox) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      out[a] = an[a] > op.prm[a];
      in = in && af[a] < op.prm[a];
    }
    // outside along two axes: every axis' line misses
    const int n = out[0] + out[1] + out[2];
    *vlo = n >= 2 ? 4.0f : n ? 1.0f : -3.0f;
    *vhi = n >= 2 ? 4.0f : in ? -1.0f : 3.0f;
    return;
  }
  *vlo = -3.0f;
  *vhi = 3.0f;
  if (op.code == kTorus) return;
  // Squares: far enough from the surface that no rounding of the squares, their
  // sums and the root (a few 2^-24 of r^2) changes a comparison.
  const float rr = op.prm[0] * op.prm[0];
  const float far = rr * 1.00002f + 1.0e-30f, near = rr * 0.99998f - 1.0e-30f;
  const float xy = an[0] * an[0] + an[1] * an[1];
  if (op.code == kSphere) {
    const float xz = an[0] * an[0] + an[2] * an[2], yz = an[1] * an[1] + an[2] * an[2];
    if (xy > far && xz > far && yz > far)
      *vlo = *vhi = 4.0f;
    else if (xy + an[2] * an[2] > far)
      *vlo = 1.0f;
    else if ((af[0] * af[0] + af[1] * af[1]) + af[2] * af[2] < near)
      *vhi = -1.0f;
  } else {  // kCylinder
    const bool above = an[2] > op.prm[1], beside = xy > far;
    if (above && beside)
      *vlo = *vhi = 4.0f;
    else if (above || beside)
      *vlo = 1.0f;
    else if (op.prm[0] > 0.0f && af[2] < op.prm[1] && af[0] * af[0] + af[1] * af[1] < near)
      *vhi = -1.0f;
  }
}

template <bool kDirected>
__device__ __forceinline__ void value_interval(const DevOp& op, const float* cl, const float* ch,
                                               float* vlo, float* vhi) {
  if constexpr (kDirected)
    directed_interval(op, cl, ch, vlo, vhi);
  else
    op_interval(op, cl, ch, vlo, vhi);
}

// Scopes that hold the whole program (a recentring wrapper): as many as open
// it and close it together.  The callers give boxes and points inside them,
// and walk the operations after their openings, with them already open.
__device__ __forceinline__ int leading_scopes(OpsPtr ops, int n) {
  int s = 0;
  while (2 * s < n && ops[s].code == kPushTranslate && ops[n - 1 - s].code == kPopTranslate) ++s;
  return s;
}

// Bounds of the operations [first, n) over one box [tlo, thi], the same for
// every lane of the wavefront, and those that can change a value in it: their
// indices go to `list` (LDS, ascending), and their number is returned (above
// `cap`: they do not fit, and the list is not usable).  Runs of min and
// smooth-min operands are bounded 64 at a time, one a lane, each against the
// running upper bound before it.
template <bool kStack, bool kDirected = false>
__device__ __forceinline__ int bound_box(OpsPtr ops, int first, int n, const float* tlo,
                                         const float* thi, uint16_t* list, int cap, float* out_lo,
                                         float* out_hi) {
  const int lane = __lane_id();
  Bounds<kStack> B;
  ScopeStack scopes;
  float cl[3] = {tlo[0], tlo[1], tlo[2]}, ch[3] = {thi[0], thi[1], thi[2]};
  int count = 0;
  for (int base = first; base < n; base += 64) {
    // One operation a lane (the last one again past the end).
    const int j = base + lane < n ? base + lane : n - 1;
    const DevOp mine = load_op(ops, j);
    const int e = n - base < 64 ? n - base : 64;
    const uint64_t run = __ballot(base + lane < n && mine.code <= kCylinder &&
                                  (mine.combine == kMin || mine.combine == kSmooth));
    int p = 0;
    while (p < e) {
      const uint64_t from = run >> p;
      if (from & 1ull) {
        const int m = ~from ? static_cast<int>(__builtin_ctzll(~from)) : 64;
        const bool in = lane >= p && lane < p + m;
        float vlo = kNoBound, vhi = kNoBound;
        if (in) value_interval<kDirected>(mine, cl, ch, &vlo, &vhi);
        const bool smooth = mine.combine == kSmooth;
        const float T = fminf(B.hi, wave_min_before(vhi));
        const bool kept = in && !(smooth ? smooth_inactive(vlo - T, mine.k) : vlo > T);
        const uint64_t keep = __ballot(kept);
        if (kept) {
          const int at = count + static_cast<int>(__popcll(keep & ((1ull << lane) - 1ull)));
          if (at < cap) list[at] = static_cast<uint16_t>(j);
        }
        count += static_cast<int>(__popcll(keep));
        B.hi = fminf(B.hi, wave_min(vhi));
        B.lo = fminf(B.lo, wave_min(kept ? vlo : kNoBound));
        // A chain of smooth minima of values that are at least x stays above
        // x less the largest blend width: a step from x - d takes off
        // (k - d)^2 / 4k, less than the k - d that is left.
        if (__ballot(kept && smooth)) {
          const float kmax = -wave_min(kept && smooth ? -mine.k : 0.0f);
          B.lo -= kmax + 1.0e-4f * (kmax + fmaxf(__builtin_fabsf(B.lo), __builtin_fabsf(B.hi)));
        }
        p += m;
        continue;
      }
      const int i = base + p;
      const DevOp op = load_op(ops, i);
      ++p;
      if (op.code <= kCylinder) {
        float vlo, vhi;
        uint64_t matters;
        value_interval<kDirected>(op, cl, ch, &vlo, &vhi);
        if (!B.join(op.combine, op.k, vlo, vhi, true, &matters)) continue;
      } else if (op.code == kPushTranslate) {
        scopes.push(i);
        enter_scope(ops, i, cl, ch);
      } else if (op.code == kPopTranslate) {
        if (scopes.depth == 0) continue;  // a leading scope's end, at the program's end
        scopes.pop();
        restore_scopes(ops, scopes, tlo, thi, cl, ch);
      } else if (kStack) {
        B.operate(op.code, op.k);
      }
      if (lane == 0 && count < cap) list[count] = static_cast<uint16_t>(i);
      ++count;
    }
  }
  *out_lo = B.lo;
  *out_hi = B.hi;
  return count;
}

// Bounds of the program over each lane's own box [blo, bhi] (`active` false:
// the lane has none), walking the m operations of `list` (null: the operations
// [first, first + m)).  With a list, the operations that matter to no lane are
// taken out of it, and mask[j] names the lanes that the j-th remaining one
// matters to.  Returns the number of operations left.
template <bool kStack, bool kDirected = false>
__device__ __forceinline__ int bound_lanes(OpsPtr ops, int first, int m, const float* blo,
                                           const float* bhi, bool active, uint16_t* list,
                                           uint64_t* mask, float* out_lo, float* out_hi) {
  const int lane = __lane_id();
  Bounds<kStack> B;
  ScopeStack scopes;
  float cl[3] = {blo[0], blo[1], blo[2]}, ch[3] = {bhi[0], bhi[1], bhi[2]};
  // The list is rewritten 64 entries at a time, from registers, one entry a
  // lane: behind the entries read so far, which `mine` holds.
  int count = 0, mine = 0, my_op = 0;
  uint64_t my_mask = 0;
  for (int j = 0; j < m; ++j) {
    if ((j & 63) == 0) mine = list ? (j + lane < m ? list[j + lane] : 0) : first + j + lane;
    const int i = __builtin_amdgcn_readlane(mine, j & 63);
    const DevOp op = load_op(ops, i);
    uint64_t matters = ~0ull;
    if (op.code <= kCylinder) {
      float vlo, vhi;
      value_interval<kDirected>(op, cl, ch, &vlo, &vhi);
      if (!B.join(op.combine, op.k, vlo, vhi, active, &matters)) continue;
    } else if (op.code == kPushTranslate) {
      scopes.push(i);
      enter_scope(ops, i, cl, ch);
    } else if (op.code == kPopTranslate) {
      if (scopes.depth == 0) continue;
      scopes.pop();
      restore_scopes(ops, scopes, blo, bhi, cl, ch);
    } else if (kStack) {
      B.operate(op.code, op.k);
    }
    if (lane == (count & 63)) {
      my_op = i;
      my_mask = matters;
    }
    ++count;
    if (list && (count & 63) == 0) {
      list[count - 64 + lane] = static_cast<uint16_t>(my_op);
      mask[count - 64 + lane] = my_mask;
    }
  }
  if (list && lane < (count & 63)) {
    list[(count & ~63) + lane] = static_cast<uint16_t>(my_op);
    mask[(count & ~63) + lane] = my_mask;
  }
  *out_lo = B.lo;
  *out_hi = B.hi;
  return count;
}

__device__ __forceinline__ float flip_sign(float x, uint32_t bit) {
  return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, x) ^ bit);
}

// sdf_eval at K points a lane (inside the leading scopes) over the operations
// named by `list` (m of them; list null: the operations [first, first + m)),
// without those whose mask has none of the bits of `bricks`.  All arguments
// but the points are the same for every lane.  The K points share each
// operation's load and dispatch, whose scalar work and latency are otherwise
// as long as one point's arithmetic.
template <int K, bool kStack>
__device__ __forceinline__ void sdf_eval_list(OpsPtr ops, int first, const uint16_t* list,
                                              const uint64_t* mask, uint64_t bricks, int m,
                                              const float (&p)[K][3], float (&top)[K]) {
  const int lane = __lane_id();
  ShiftStack st[K];
  float c[K][3];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    top[k] = kNoBound;  // min(kNoBound, v) is v: the first push is read as a min
#pragma unroll
    for (int i = 0; i < kMaxValueStack; ++i) st[k].v[i] = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) c[k][a] = p[k][a];
  }
  ScopeStack scopes;
  bool have_top = false;
  for (int base = 0; base < m; base += 64) {
    int mine = first + base + lane;
    bool use = base + lane < m;
    if (list && use) {
      mine = list[base + lane];
      use = (mask[base + lane] & bricks) != 0ull;
    }
    uint64_t todo = __ballot(use);
    while (todo) {
      const int i = __builtin_amdgcn_readlane(mine, static_cast<int>(__builtin_ctzll(todo)));
      todo &= todo - 1;
      const DevOp op = load_op(ops, i);
      const uint32_t code = op.code;
      if (code <= kCylinder) {
        float q[K][3], v[K];
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) q[k][a] = c[k][a] - op.off[a];  // (x - 0 is x)
        prim_values(code, op.prm, q, v);
        const uint32_t mode = op.combine;
        if (kStack && mode == kPush) {
#pragma unroll
          for (int k = 0; k < K; ++k) {
            if (have_top) st[k].push(top[k]);
            top[k] = v[k];
          }
          have_top = true;
        } else if (mode == kMin || (!kStack && mode == kPush)) {
#pragma unroll
          for (int k = 0; k < K; ++k) top[k] = fminf(top[k], v[k]);
        } else if (mode == kSmooth) {
#pragma unroll
          for (int k = 0; k < K; ++k) top[k] = smooth_min(top[k], v[k], op.k);
        } else {
          // max(top, v), max(v, -top) or max(top, -v)
          const uint32_t nt = mode == kDiff ? 0x80000000u : 0u;
          const uint32_t nv = mode == kDiffRev ? 0x80000000u : 0u;
#pragma unroll
          for (int k = 0; k < K; ++k)
            top[k] = fmaxf(flip_sign(top[k], nt), flip_sign(v[k], nv));
        }
      } else if (code == kPushTranslate) {
        scopes.push(i);
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - op.off[a];
      } else if (code == kPopTranslate) {
        if (scopes.depth == 0) continue;
        scopes.pop();
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) c[k][a] = p[k][a];
        for (int s = 0; s < scopes.depth; ++s) {
          const int o = scopes.at(s);
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - ops[o].off[a];
        }
      } else if (kStack) {
        const uint32_t nw = code == kDifference ? 0x80000000u : 0u;
        const uint32_t nt = code == kDifferenceRev ? 0x80000000u : 0u;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const float w = st[k].pop();
          if (code == kUnion)
            top[k] = fminf(w, top[k]);
          else if (code == kSmoothUnion)
            top[k] = smooth_min(w, top[k], op.k);
          else  // max(w, t), max(t, -w) or max(w, -t)
            top[k] = fmaxf(flip_sign(w, nw), flip_sign(top[k], nt));
        }
      }
    }
  }
}

// sdf_eval_vector (Directed values) over a list of operations, as sdf_eval_list.
template <int K, bool kStack>
__device__ __forceinline__ void sdf_eval_vector_list(OpsPtr ops, int first, const uint16_t* list,
                                                     const uint64_t* mask, uint64_t bricks, int m,
                                                     const float (&p)[K][3], float (&top)[K][3]) {
  const int lane = __lane_id();
  ShiftStack st[K][3];
  float c[K][3];
#pragma unroll
  for (int k = 0; k < K; ++k)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      top[k][a] = __builtin_inff();  // min(inf, v) is v: the first push is read as a min
      c[k][a] = p[k][a];
#pragma unroll
      for (int i = 0; i < kMaxValueStack; ++i) st[k][a].v[i] = 0.0f;
    }
  ScopeStack scopes;
  bool have_top = false;
  for (int base = 0; base < m; base += 64) {
    int mine = first + base + lane;
    bool use = base + lane < m;
    if (list && use) {
      mine = list[base + lane];
      use = (mask[base + lane] & bricks) != 0ull;
    }
    uint64_t todo = __ballot(use);
    while (todo) {
      const int i = __builtin_amdgcn_readlane(mine, static_cast<int>(__builtin_ctzll(todo)));
      todo &= todo - 1;
      const DevOp op = load_op(ops, i);
      const uint32_t code = op.code;
      if (code <= kCylinder) {
        const uint32_t mode = op.combine;
        const bool least = mode == kMin || (!kStack && mode == kPush);
        const uint32_t nt = mode == kDiff ? 0x80000000u : 0u;
        const uint32_t nv = mode == kDiffRev ? 0x80000000u : 0u;
        if (kStack && mode == kPush && have_top) {
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) st[k][a].push(top[k][a]);
        }
        if (mode == kPush) have_top = true;
#pragma unroll
        for (int k = 0; k < K; ++k) {
          float v[3];
          prim_vector(code, op.prm, c[k][0] - op.off[0], c[k][1] - op.off[1],
                      c[k][2] - op.off[2], v);  // (x - 0 is x)
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            // min, or max(top, v), max(v, -top), max(top, -v)
            if (kStack && mode == kPush)
              top[k][a] = v[a];
            else if (least)
              top[k][a] = fminf(top[k][a], v[a]);
            else
              top[k][a] = fmaxf(flip_sign(top[k][a], nt), flip_sign(v[a], nv));
          }
        }
      } else if (code == kPushTranslate) {
        scopes.push(i);
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - op.off[a];
      } else if (code == kPopTranslate) {
        if (scopes.depth == 0) continue;
        scopes.pop();
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) c[k][a] = p[k][a];
        for (int s = 0; s < scopes.depth; ++s) {
          const int o = scopes.at(s);
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - ops[o].off[a];
        }
      } else if (kStack) {
        const uint32_t nw = code == kDifference ? 0x80000000u : 0u;
        const uint32_t nt = code == kDifferenceRev ? 0x80000000u : 0u;
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
          for (int a = 0; a < 3; ++a) {
            const float w = st[k][a].pop();
            // min, or max(w, t), max(t, -w), max(w, -t)
            top[k][a] = code == kUnion ? fminf(w, top[k][a])
                                       : fmaxf(flip_sign(w, nw), flip_sign(top[k][a], nt));
          }
      }
    }
  }
}

// An operation held by lane `from` of the wavefront.
__device__ __forceinline__ DevOp lane_op(const DevOp& mine, int from) {
  auto f = [&](float x) {
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), from));
  };
  DevOp o;
  o.code = __builtin_amdgcn_readlane(mine.code, from);
  o.combine = __builtin_amdgcn_readlane(mine.combine, from);
  o.translated = 0;
  o.k = f(mine.k);
#pragma unroll
  for (int a = 0; a < 4; ++a) o.prm[a] = f(mine.prm[a]);
#pragma unroll
  for (int a = 0; a < 3; ++a) o.off[a] = f(mine.off[a]);
  o.off[3] = 0.0f;
  return o;
}

// sdf_eval of a bounded program at K points a lane, for a wavefront whose
// points lie close together: it reads 64 operations
// at once, one a lane, bounds the runs of min and smooth-min operands over the
// box of its points, and evaluates out of those registers what can change a
// value.  `head`: the first 64 operations (lane_ops), which the caller reads
// when it has something to wait for.  Every lane takes part.
__device__ __forceinline__ DevOp lane_ops(OpsPtr ops, int base, int n) {
  const int j = base + static_cast<int>(__lane_id());
  return load_op(ops, j < n ? j : n - 1);
}

template <int K, bool kStack>
__device__ __forceinline__ void sdf_eval_near(OpsPtr ops, int n, const DevOp& head,
                                              const float (&base_p)[K][3], float (&top)[K]) {
  const int lane = __lane_id();
  float c[K][3], cl[3], ch[3];
  auto box = [&] {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      float lo = c[0][a], hi = c[0][a];
#pragma unroll
      for (int k = 1; k < K; ++k) {
        lo = fminf(lo, c[k][a]);
        hi = fmaxf(hi, c[k][a]);
      }
      cl[a] = wave_min(lo);
      ch[a] = -wave_min(-hi);
    }
  };
  ShiftStack st[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    top[k] = kNoBound;
#pragma unroll
    for (int i = 0; i < kMaxValueStack; ++i) st[k].v[i] = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a) c[k][a] = base_p[k][a];
  }
  box();
  ScopeStack scopes;
  bool have_top = false;
  for (int base = 0; base < n; base += 64) {
    const DevOp mine = base == 0 ? head : lane_ops(ops, base, n);
    const int e = n - base < 64 ? n - base : 64;
    const uint64_t run = __ballot(base + lane < n && mine.code <= kCylinder &&
                                  (mine.combine == kMin || mine.combine == kSmooth));
    int p = 0;
    while (p < e) {
      const uint64_t from = run >> p;
      uint64_t todo = 1ull << p;
      int m = 1;
      if (from & 1ull) {
        m = ~from ? static_cast<int>(__builtin_ctzll(~from)) : 64;
        const bool in = lane >= p && lane < p + m;
        float vlo = kNoBound, vhi = kNoBound;
        if (in) op_interval(mine, cl, ch, &vlo, &vhi);
        // as bound_box, from the greatest running value itself
        float most = top[0];
#pragma unroll
        for (int k = 1; k < K; ++k) most = fmaxf(most, top[k]);
        const float T = fminf(-wave_min(-most), wave_min_before(vhi));
        todo = __ballot(in && !(mine.combine == kSmooth ? smooth_inactive(vlo - T, mine.k)
                                                        : vlo > T));
      }
      p += m;
      for (; todo; todo &= todo - 1) {
        const int j = static_cast<int>(__builtin_ctzll(todo));
        const DevOp op = lane_op(mine, j);
        if (op.code <= kCylinder) {
          float q[K][3], v[K];
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) q[k][a] = c[k][a] - op.off[a];  // (x - 0 is x)
          prim_values(op.code, op.prm, q, v);
          const uint32_t mode = op.combine;
          if (kStack && mode == kPush && have_top) {
#pragma unroll
            for (int k = 0; k < K; ++k) st[k].push(top[k]);
          }
          if (mode == kPush) have_top = true;
          // max(top, v), max(v, -top) or max(top, -v)
          const uint32_t nt = mode == kDiff ? 0x80000000u : 0u;
          const uint32_t nv = mode == kDiffRev ? 0x80000000u : 0u;
#pragma unroll
          for (int k = 0; k < K; ++k)
            top[k] = mode == kPush     ? v[k]
                     : mode == kMin    ? fminf(top[k], v[k])
                     : mode == kSmooth ? smooth_min(top[k], v[k], op.k)
                                       : fmaxf(flip_sign(top[k], nt), flip_sign(v[k], nv));
        } else if (op.code == kPushTranslate) {
          scopes.push(base + j);
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - op.off[a];
          box();
        } else if (op.code == kPopTranslate) {
          scopes.pop();
#pragma unroll
          for (int k = 0; k < K; ++k)
#pragma unroll
            for (int a = 0; a < 3; ++a) c[k][a] = base_p[k][a];
          for (int s = 0; s < scopes.depth; ++s) {
            const int o = scopes.at(s);
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
              for (int a = 0; a < 3; ++a) c[k][a] = c[k][a] - ops[o].off[a];
          }
          box();
        } else if (kStack) {
          const uint32_t nw = op.code == kDifference ? 0x80000000u : 0u;
          const uint32_t nt = op.code == kDifferenceRev ? 0x80000000u : 0u;
#pragma unroll
          for (int k = 0; k < K; ++k) {
            const float w = st[k].pop();
            top[k] = op.code == kUnion         ? fminf(w, top[k])
                     : op.code == kSmoothUnion ? smooth_min(w, top[k], op.k)
                                               // max(w, t), max(t, -w) or max(w, -t)
                                               : fmaxf(flip_sign(w, nw), flip_sign(top[k], nt));
          }
        }
      }
    }
  }
}

// Whether a tile of whose n_ops operations m matter, too many for its list, is
// better evaluated by sdf_eval_near: where nearly all matter throughout the tile
// they also do in a wavefront's share of it, and bounding them again is lost.
__device__ __forceinline__ bool prunes_near(int m, int n_ops) { return m <= n_ops - n_ops / 64; }

// A barrier for what the tile's wavefronts exchange in LDS: __syncthreads
// would also wait for the samples on their way to memory (two microseconds a
// tile).
template <int W>
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if (W > 1) __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Stores the sign words of a 16^3-sample tile at sample s0 (tile tx along x)
// from its 64 blocks' bits (4^3 samples each, x fastest): 16 bits of each row,
// four from each block along x.
__device__ __forceinline__ void store_tile_signs(const CellSpace& C, const uint64_t* s_sign,
                                                 const int32_t* s0, uint32_t tx, int thread,
                                                 int threads) {
  const int32_t ny = static_cast<int32_t>(C.ny), nz = static_cast<int32_t>(C.nz);
  uint16_t* S = reinterpret_cast<uint16_t*>(const_cast<uint64_t*>(C.signs));
  for (int r = thread; r < 256; r += threads) {
    const int ry = r & 15, rz = r >> 4;
    const int32_t y = s0[1] + ry, z = s0[2] + rz;
    if (y >= ny || z >= nz) continue;
    const int b0 = (rz >> 2) * 16 + (ry >> 2) * 4;
    const int sh = 16 * (rz & 3) + 4 * (ry & 3);
    uint32_t bits = 0;
#pragma unroll
    for (int bx = 0; bx < 4; ++bx)
      bits |= static_cast<uint32_t>((s_sign[b0 + bx] >> sh) & 0xFull) << (4 * bx);
    S[(static_cast<int64_t>(z) * ny + y) * (C.sign_pitch >> 4) + tx] = static_cast<uint16_t>(bits);
  }
}

// ---------------------------------------------------------------------------
// Evaluation with an error bound (sdf_eval_bound) over a list of operations.
// ---------------------------------------------------------------------------

// The operations of a bounded program that matter to sdf_eval_bound at points
// of the box [blo, bhi], for balls of radius `widen` at most: bound_box's, and
// also the smooth-min operands whose blend its error bound might count (within
// the blend width, the ball and the errors of either operand, which `mag`, a
// bound of every coordinate and parameter, bounds in turn).  Returns their
// number (above `cap`: they do not fit).  *floor_e receives the greatest error
// bound of any primitive at a point of the box.
__device__ __forceinline__ int certify_list(OpsPtr ops, int n, const float* blo, const float* bhi,
                                            float widen, float mag, uint16_t* list, int cap,
                                            float* floor_e) {
  constexpr float u = 5.9604645e-08f;  // 2^-24
  const int lane = __lane_id();
  ScopeStack scopes;
  float cl[3] = {blo[0], blo[1], blo[2]}, ch[3] = {bhi[0], bhi[1], bhi[2]};
  float pe = 0.0f;  // bound of the rounding of the box's translated points
  float top = kNoBound;  // upper bound of the running value of the current run
  float worst = 0.0f;
  int count = 0;
  // Twice the errors of two operands, a primitive's being at most 64 u (mag +
  // 2 widen) and each blend adding at most u (10 k + 4 (mag + 2 widen)) to the
  // running one, and the rounding of the operands' difference.
  auto room = [&](float k) {
    const float w = mag + 2.0f * widen;
    return 2.0f * u * (128.0f * w + static_cast<float>(n) * (10.0f * k + 4.0f * w)) + 16.0f * u * w;
  };
  auto far_of = [&](const DevOp& op) {  // greatest |q_c| over the box, and the primitive's error
    float q = 0.0f;
#pragma unroll
    for (int a = 0; a < 3; ++a)
      q = fmaxf(q, fmaxf(-(cl[a] - op.off[a]), ch[a] - op.off[a]));
    const float qe = op.translated ? pe + u * (q + widen + pe) : pe;
    const float qmax = q + widen + qe;
    const float pm = __builtin_fabsf(op.prm[0]) + __builtin_fabsf(op.prm[1]) +
                     __builtin_fabsf(op.prm[2]) + __builtin_fabsf(op.prm[3]);
    return 1.7320509f * qe + 16.0f * u * (1.7320509f * qmax + pm);
  };
  for (int base = 0; base < n; base += 64) {
    const int j = base + lane < n ? base + lane : n - 1;
    const DevOp mine = load_op(ops, j);
    const int e = n - base < 64 ? n - base : 64;
    const uint64_t run = __ballot(base + lane < n && mine.code <= kCylinder &&
                                  (mine.combine == kMin || mine.combine == kSmooth));
    int p = 0;
    while (p < e) {
      const uint64_t from = run >> p;
      if (from & 1ull) {
        const int m = ~from ? static_cast<int>(__builtin_ctzll(~from)) : 64;
        const bool in = lane >= p && lane < p + m;
        float vlo = kNoBound, vhi = kNoBound, err = 0.0f;
        if (in) {
          op_interval(mine, cl, ch, &vlo, &vhi);
          err = far_of(mine);
        }
        const float T = fminf(top, wave_min_before(vhi));
        const float gap = (vlo - T) * (1.0f - 8.0f * u);
        const bool idle = mine.combine == kSmooth
                              ? gap >= (mine.k + 2.0f * widen + room(mine.k)) * (1.0f + 8.0f * u)
                              : vlo > T;
        const bool kept = in && !idle;
        const uint64_t keep = __ballot(kept);
        if (kept) {
          const int at = count + static_cast<int>(__popcll(keep & ((1ull << lane) - 1ull)));
          if (at < cap) list[at] = static_cast<uint16_t>(j);
        }
        count += static_cast<int>(__popcll(keep));
        top = fminf(top, wave_min(vhi));
        worst = fmaxf(worst, -wave_min(-err));
        p += m;
        continue;
      }
      const int i = base + p;
      const DevOp op = load_op(ops, i);
      ++p;
      if (op.code <= kCylinder) {
        float vlo, vhi;
        op_interval(op, cl, ch, &vlo, &vhi);
        worst = fmaxf(worst, far_of(op));
        top = op.combine == kPush ? vhi : kNoBound;  // (after a max: not bounded here)
      } else if (op.code == kPushTranslate) {
        scopes.push(i);
        enter_scope(ops, i, cl, ch);
        float q = 0.0f;
#pragma unroll
        for (int a = 0; a < 3; ++a) q = fmaxf(q, fmaxf(-cl[a], ch[a]));
        pe = pe + u * (q + widen + pe);
      } else if (op.code == kPopTranslate) {
        scopes.pop();
        restore_scopes(ops, scopes, blo, bhi, cl, ch);
        // (pe stays at the inner scope's, which is no smaller)
      } else {
        top = kNoBound;  // a binary operator's value: not bounded here
      }
      if (lane == 0 && count < cap) list[count] = static_cast<uint16_t>(i);
      ++count;
    }
  }
  *floor_e = worst;
  return count;
}

// sdf_eval_bound over the m operations of `list` (certify_list's): its value,
// and two bounds of its error bound, from the listed operations alone (*e0) and
// with every operand's error at least floor_e (*e1).
template <bool kStack>
__device__ __forceinline__ float eval_bound_list(OpsPtr ops, const uint16_t* list, int m, float px,
                                                 float py, float pz, float widen, float floor_e,
                                                 float* e0, float* e1) {
  constexpr float u = 5.9604645e-08f;  // 2^-24
  const int lane = __lane_id();
  float top = 0.0f, a0 = 0.0f, a1 = 0.0f;
  ShiftStack st, s0, s1;
#pragma unroll
  for (int i = 0; i < kMaxValueStack; ++i) st.v[i] = s0.v[i] = s1.v[i] = 0.0f;
  float c[3] = {px, py, pz}, pe = 0.0f;
  ScopeStack scopes;
  bool have_top = false;
  auto moved = [&](const float* q, float e) {
    return e + u * (bound_max3(__builtin_fabsf(q[0]), __builtin_fabsf(q[1]), __builtin_fabsf(q[2])) +
                    widen + e);
  };
  auto blend = [&](float a, float ea, float b, float eb, float k) {
    float e = fmaxf(ea, eb);
    if (__builtin_fabsf(a - b) < k + 2.0f * widen + 2.0f * (ea + eb) +
                                     u * (__builtin_fabsf(a) + __builtin_fabsf(b))) {
      const float mg = fminf(__builtin_fabsf(a), __builtin_fabsf(b)) + widen + e;
      e += 8.0f * u * k + 2.0f * u * (mg + k);
    }
    return e;
  };
  for (int base = 0; base < m; base += 64) {
    const int mine = base + lane < m ? list[base + lane] : 0;
    const int e = m - base < 64 ? m - base : 64;
    for (int j = 0; j < e; ++j) {
      const int i = __builtin_amdgcn_readlane(mine, j);
      const DevOp op = load_op(ops, i);
      if (op.code <= kCylinder) {
        float q[1][3], v[1];
#pragma unroll
        for (int a = 0; a < 3; ++a) q[0][a] = c[a] - op.off[a];
        const float qe = op.translated ? moved(q[0], pe) : pe;
        prim_values(op.code, op.prm, q, v);
        const float qmax =
            bound_max3(__builtin_fabsf(q[0][0]), __builtin_fabsf(q[0][1]),
                       __builtin_fabsf(q[0][2])) + widen + qe;
        const float pm = __builtin_fabsf(op.prm[0]) + __builtin_fabsf(op.prm[1]) +
                         __builtin_fabsf(op.prm[2]) + __builtin_fabsf(op.prm[3]);
        const float ev = 1.7320509f * qe + 16.0f * u * (1.7320509f * qmax + pm);
        const float ev1 = fmaxf(ev, floor_e);
        if (op.combine == kPush) {
          if (kStack && have_top) {
            st.push(top);
            s0.push(a0);
            s1.push(a1);
          }
          top = v[0];
          a0 = ev;
          a1 = ev1;
          have_top = true;
        } else if (op.combine == kSmooth) {
          a0 = blend(top, a0, v[0], ev, op.k);
          a1 = blend(top, a1, v[0], ev1, op.k);
          top = smooth_min(top, v[0], op.k);
        } else {
          if (op.combine == kMin)
            top = fminf(top, v[0]);
          else if (op.combine == kMax)
            top = fmaxf(top, v[0]);
          else if (op.combine == kDiff)
            top = fmaxf(v[0], -top);
          else
            top = fmaxf(top, -v[0]);
          a0 = fmaxf(a0, ev);
          a1 = fmaxf(a1, ev1);
        }
      } else if (op.code == kPushTranslate) {
        scopes.push(i);
#pragma unroll
        for (int a = 0; a < 3; ++a) c[a] = c[a] - op.off[a];
        pe = moved(c, pe);
      } else if (op.code == kPopTranslate) {
        scopes.pop();
        c[0] = px;
        c[1] = py;
        c[2] = pz;
        pe = 0.0f;
        for (int s = 0; s < scopes.depth; ++s) {
          const int o = scopes.at(s);
#pragma unroll
          for (int a = 0; a < 3; ++a) c[a] = c[a] - ops[o].off[a];
          pe = moved(c, pe);
        }
      } else if (kStack) {
        const float w = st.pop(), w0 = s0.pop(), w1 = s1.pop();
        if (op.code == kSmoothUnion) {
          a0 = blend(w, w0, top, a0, op.k);
          a1 = blend(w, w1, top, a1, op.k);
          top = smooth_min(w, top, op.k);
        } else {
          if (op.code == kUnion)
            top = fminf(w, top);
          else if (op.code == kIntersection)
            top = fmaxf(w, top);
          else if (op.code == kDifference)
            top = fmaxf(top, -w);
          else
            top = fmaxf(w, -top);
          a0 = fmaxf(w0, a0);
          a1 = fmaxf(w1, a1);
        }
      }
    }
  }
  *e0 = a0 * 1.001f;
  *e1 = a1 * 1.001f;
  return top;
}

}  // namespace iso
