// Feature placement of dual contouring on the device: TangentPlanes
// classification in f32 and the QEF solve of MinimiseQEF through the SVD of
// the 8 x 3 normal matrix in f64.
//
// Bit-identical results with the reference require its exact arithmetic, so
// every step follows feature/mod.rs:91-148, feature/qef.rs:36-68 and
// math/svd.rs:25-84, 130-972 operation for operation (the library is built
// with -ffp-contract=off; f64 sqrt and division are correctly rounded).  The
// one liberty taken is data movement: the reference copies the active column
// window into scratch matrices before each QR step, here the step works on
// the window in place, which performs the same arithmetic on the same values.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

namespace iso {
namespace qef {

constexpr int kRows = 8;     // dual contouring: the 8 cell corners
constexpr int kMaxRows = 12;  // extended marching cubes: up to 12 edge crossings

struct Vec3f {
  float x, y, z;
};

__device__ __forceinline__ float dot3(Vec3f a, Vec3f b) {
  return (a.x * b.x + a.y * b.y) + a.z * b.z;  // vector.rs:240-242, 290-292
}

__device__ __forceinline__ Vec3f cross3(Vec3f a, Vec3f b) {
  return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// Vec3::normalised().unwrap_or_default() (vector.rs:135-144).
__device__ __forceinline__ Vec3f normalised_or_zero(Vec3f v) {
  const float l = __builtin_sqrtf((v.x * v.x + v.y * v.y) + v.z * v.z);
  if (__builtin_fabsf(l) < 1.1920929e-07f) return {0.0f, 0.0f, 0.0f};
  return {v.x / l, v.y / l, v.z / l};
}

// The SVD of a rows x 3 matrix (rows <= R): every loop over rows runs to
// `rows`, so the arithmetic is that of the reference's rows-row matrix.
//
// One thread's solve is a serial chain of f64 operations, and latency bounds
// it: a launch has about one wavefront for each SIMD.  So indices are constants
// once the loops are unrolled (the column window is a template argument, a
// run-time column becomes a choice between constants), and cases that differ
// in their operands choose those first and share one chain: the feature pass
// of 128^3 dual contouring over 32 boxes takes 37 us, with run-time columns and
// a division in every branch 48.
template <int R>
struct SvdT {
  double u[R][3];
  double v[3][3];
  double d[3];
  int rows;
};

// Householder reflection of the n <= N entries x[0], x[stride], ... (svd.rs:251-293).
template <int N, int stride>
__device__ __forceinline__ double householder(double* x, int n) {
  double tau = 0.0;
  if (n > 1) {
    double xnorm;
    if (n == 2) {
      xnorm = __builtin_fabs(x[stride]);
    } else {
      double scl = 0.0, ssq = 1.0;
#pragma unroll
      for (int i = 1; i < N; ++i) {
        if (i >= n) continue;
        const double a = __builtin_fabs(x[i * stride]);
        if (a != 0.0) {  // (one division for both cases)
          const bool up = scl < a;
          const double r = (up ? scl : a) / (up ? a : scl);
          ssq = up ? 1.0 + ssq * r * r : ssq + r * r;
          scl = up ? a : scl;
        }
      }
      xnorm = scl * __builtin_sqrt(ssq);
    }
    if (xnorm != 0.0) {
      const double alpha = x[0];
      double beta = __builtin_sqrt(alpha * alpha + xnorm * xnorm);
      if (alpha >= 0.0) beta = -beta;
      tau = (beta - alpha) / beta;
      const double scl = 1.0 / (alpha - beta);
      x[0] = beta;
#pragma unroll
      for (int i = 1; i < N; ++i)
        if (i < n) x[i * stride] *= scl;
    }
  }
  return tau;
}

// Step i of the bidiagonal factorisation (svd.rs:149-249).
template <int R, int i>
__device__ __forceinline__ void bidiagonalise_step(double m[R][3], double tau_u[3], double tau_v[2],
                                                   int rows) {
  double tau = householder<R - i, 3>(&m[i][i], rows - i);
  tau_u[i] = tau;
  if constexpr (i + 1 < 3) {
    if (tau != 0.0) {
#pragma unroll
      for (int x = i + 1; x < 3; ++x) {
        double wx = m[i][x];
#pragma unroll
        for (int y = i + 1; y < R; ++y)
          if (y < rows) wx += m[y][x] * m[y][i];
        const double tw = tau * wx;
        m[i][x] -= tw;
#pragma unroll
        for (int y = i + 1; y < R; ++y)
          if (y < rows) m[y][x] -= tw * m[y][i];
      }
    }
    tau = householder<2 - i, 1>(&m[i][i + 1], 2 - i);
    tau_v[i] = tau;
    if (tau != 0.0) {
#pragma unroll
      for (int y = i + 1; y < R; ++y) {
        if (y >= rows) continue;
        double wy = m[y][i + 1];
        if constexpr (i == 0) wy += m[y][i + 2] * m[i][i + 2];
        const double tw = tau * wy;
        m[y][i + 1] -= tw;
        if constexpr (i == 0) m[y][i + 2] -= tw * m[i][i + 2];
      }
    }
  }
}
template <int R>
__device__ __forceinline__ void bidiagonalise(double m[R][3], double tau_u[3], double tau_v[2],
                                              int rows) {
  bidiagonalise_step<R, 0>(m, tau_u, tau_v, rows);
  bidiagonalise_step<R, 1>(m, tau_u, tau_v, rows);
  bidiagonalise_step<R, 2>(m, tau_u, tau_v, rows);
}

// Accumulates the reflections into U and V (svd.rs:295-410).
template <int R>
__device__ __forceinline__ void unpack(double u[R][3], double v[3][3], double tau_u[3],
                                       double tau_v[2], int rows) {
#pragma unroll
  for (int i = 0; i < 3; ++i)
#pragma unroll
    for (int j = 0; j < 3; ++j) v[i][j] = i == j ? 1.0 : 0.0;
#pragma unroll
  for (int i = 1; i >= 0; --i) {
    const double tau = tau_v[i];
    if (tau != 0.0) {
#pragma unroll
      for (int x = i + 1; x < 3; ++x) {
        double wx = v[i + 1][x];
#pragma unroll
        for (int y = i + 2; y < 3; ++y) wx += v[y][x] * u[i][y];
        const double tw = tau * wx;
        v[i + 1][x] -= tw;
#pragma unroll
        for (int y = i + 2; y < 3; ++y) v[y][x] -= tw * u[i][y];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) tau_v[i] = u[i][i + 1];
#pragma unroll
  for (int i = 2; i >= 0; --i) {
    const double tau = tau_u[i];
    tau_u[i] = u[i][i];
    if (tau == 0.0) {
      u[i][i] = 1.0;
      if (i < 2) {
        u[i][2] = 0.0;
        if (i < 1) u[i][1] = 0.0;
      }
#pragma unroll
      for (int y = i + 1; y < R; ++y)
        if (y < rows) u[y][i] = 0.0;
    } else {
#pragma unroll
      for (int x = i + 1; x < 3; ++x) {
        double wx = 0.0;
#pragma unroll
        for (int y = i + 1; y < R; ++y)
          if (y < rows) wx += u[y][x] * u[y][i];
        const double tw = tau * wx;
        u[i][x] = -tw;
#pragma unroll
        for (int y = i + 1; y < R; ++y)
          if (y < rows) u[y][x] -= tw * u[y][i];
      }
#pragma unroll
      for (int y = i + 1; y < R; ++y)
        if (y < rows) u[y][i] = u[y][i] * -tau;
      u[i][i] = 1.0 - tau;
    }
  }
}

// The cases of the next three differ in their operands: chosen first, each is
// one chain of divisions and square roots for the whole wavefront.
__device__ __forceinline__ void givens(double a, double b, double* c, double* s) {  // svd.rs:825-842
  const bool steep = __builtin_fabs(b) > __builtin_fabs(a);
  const double t = -(steep ? a : b) / (steep ? b : a);
  const double r = 1.0 / __builtin_sqrt(1.0 + t * t);
  const double rt = r * t;
  *c = b == 0.0 ? 1.0 : steep ? rt : r;
  *s = b == 0.0 ? 0.0 : steep ? r : rt;
}

__device__ __forceinline__ void schur(double a1, double a2, double a3, double* c, double* s) {  // svd.rs:844-865
  const double apq = a1 * a2 * 2.0;
  if (apq == 0.0) {
    *c = 1.0;
    *s = 0.0;
  } else {
    const double tau = (a2 * a2 + (a3 + a1) * (a3 - a1)) / apq;
    const double q = __builtin_sqrt(1.0 + tau * tau);
    const double r = 1.0 / (tau >= 0.0 ? tau + q : q - tau);
    const double t = tau >= 0.0 ? r : -r;
    *c = 1.0 / __builtin_sqrt(1.0 + t * t);
    *s = t * *c;
  }
}

// On the n columns from a on (svd.rs:481-493).
template <int a, int n>
__device__ __forceinline__ void chop(double tu[3], double tv[2]) {
#pragma unroll
  for (int i = a; i < a + n - 1; ++i)
    if (__builtin_fabs(tv[i]) < 1e-5 * (__builtin_fabs(tu[i]) + __builtin_fabs(tu[i + 1])))
      tv[i] = 0.0;
}

// Rotates columns p and q of the first `rows` rows by (c, s).
template <int R, int p, int q>
__device__ __forceinline__ void rotate(double m[R][3], int rows, double c, double s) {
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i >= rows) continue;
    const double mp = m[i][p], mq = m[i][q];
    m[i][p] = mp * c - mq * s;
    m[i][q] = mp * s + mq * c;
  }
}

template <int a, int b, int R>
__device__ __forceinline__ void swap_cols(double m[R][3], int rows) {
#pragma unroll
  for (int i = 0; i < R; ++i) {
    if (i >= rows) continue;
    const double t = m[i][a];
    m[i][a] = m[i][b];
    m[i][b] = t;
  }
}

// QR step on the 2-column window [a, a+1] (svd.rs:689-823).
template <int a, int R>
__device__ __forceinline__ void qr_cols2(SvdT<R>& S, double tu[3], double tv[2]) {
  double c, s;
  if (tu[a] == 0.0) {
    givens(tv[a], tu[a + 1], &c, &s);
    tu[a] = tv[a] * c - tu[a + 1] * s;
    tv[a] = tv[a] * s + tu[a + 1] * c;
    tu[a + 1] = 0.0;
    rotate<R, a, a + 1>(S.u, S.rows, c, s);
    swap_cols<a, a + 1, 3>(S.v, 3);
  } else if (tu[a + 1] == 0.0) {
    givens(tu[a], tv[a], &c, &s);
    tu[a] = tu[a] * c - tv[a] * s;
    tv[a] = 0.0;
    rotate<3, a, a + 1>(S.v, 3, c, s);
  } else {
    schur(tu[a], tv[a], tu[a + 1], &c, &s);
    double a11 = tu[a] * c - tv[a] * s;
    double a21 = -tu[a + 1] * s;
    double a12 = tu[a] * s + tv[a] * c;
    double a22 = tu[a + 1] * c;
    rotate<3, a, a + 1>(S.v, 3, c, s);
    if (a11 * a11 + a21 * a21 < a12 * a12 + a22 * a22) {
      double t = a11;
      a11 = a12;
      a12 = t;
      t = a21;
      a21 = a22;
      a22 = t;
      swap_cols<a, a + 1, 3>(S.v, 3);
    }
    givens(a11, a21, &c, &s);
    tu[a] = a11 * c - a21 * s;
    tv[a] = a12 * c - a22 * s;
    tu[a + 1] = a12 * s + a22 * c;
    rotate<R, a, a + 1>(S.u, S.rows, c, s);
  }
}

// A zero on the diagonal at `col` inside the 3-column window (svd.rs:604-641).
template <int col, int R>
__device__ __forceinline__ void qr_middle(SvdT<R>& S, double tu[3], double tv[2]) {
  double x = tv[col], y = tu[col + 1];
#pragma unroll
  for (int j = col; j < 2; ++j) {
    double c, s;
    givens(y, -x, &c, &s);
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i >= S.rows) continue;
      const double up = S.u[i][col], uq = S.u[i][j + 1];
      S.u[i][col] = up * c - uq * s;
      S.u[i][j + 1] = up * s + uq * c;
    }
    tu[j + 1] = x * s + y * c;
    if (j == col) tv[j] = x * c - y * s;
    if (j < 1) {
      const double z = tv[j + 1];
      tv[j + 1] *= c;
      x = z * -s;
      y = tu[j + 2];
    }
  }
}

// A zero at the end of the diagonal (svd.rs:643-671).
template <int R>
__device__ __forceinline__ void qr_end(SvdT<R>& S, double tu[3], double tv[2]) {
  double x = tu[1], y = tv[1];
#pragma unroll
  for (int k = 1; k >= 0; --k) {
    double c, s;
    givens(x, y, &c, &s);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double vp = S.v[i][k], vq = S.v[i][2];
      S.v[i][k] = vp * c - vq * s;
      S.v[i][2] = vp * s + vq * c;
    }
    tu[k] = x * c - y * s;
    if (k == 1) tv[k] = x * s + y * c;
    if (k > 0) {
      const double z = tv[k - 1];
      tv[k - 1] *= c;
      x = tu[k - 1];
      y = z * s;
    }
  }
}

__device__ __forceinline__ double qr_shift(const double* tu, const double* tv) {  // svd.rs:673-687
  const double ta = tu[1] * tu[1] + tv[0] * tv[0];
  const double tb = tu[2] * tu[2] + tv[1] * tv[1];
  const double tab = tu[1] * tv[1];
  const double dt = (ta - tb) / 2.0;
  const double q = __builtin_sqrt(dt * dt + tab * tab);
  const double r = tab * tab / (dt >= 0.0 ? dt + q : q - dt);
  return dt >= 0.0 ? tb - r : tb + r;
}

// Column k of a sweep over the whole matrix.
template <int k, int R>
__device__ __forceinline__ void qr_column(SvdT<R>& S, double tu[3], double tv[2], double& y,
                                          double& z, double& ak, double& bk, double& zk, double& ap,
                                          double& bp, double& aq) {
  double c, s;
  givens(y, z, &c, &s);
  rotate<3, k, k + 1>(S.v, 3, c, s);
  double bk1 = bk * c - z * s;
  double ap1 = ap * c - bp * s;
  double bp1 = ap * s + bp * c;
  const double zp1 = aq * -s;
  const double aq1 = aq * c;
  if constexpr (k > 0) tv[k - 1] = bk1;
  ak = ap1;
  bk = bp1;
  zk = zp1;
  ap = aq1;
  bp = 0.0;
  if constexpr (k < 1) bp = tv[k + 1];
  y = ak;
  z = zk;
  givens(y, z, &c, &s);
  rotate<R, k, k + 1>(S.u, S.rows, c, s);
  const double ak1 = ak * c - zk * s;
  bk1 = bk * c - ap * s;
  const double zk1 = bp * -s;
  ap1 = bk * s + ap * c;
  bp1 = bp * c;
  tu[k] = ak1;
  ak = ak1;
  bk = bk1;
  zk = zk1;
  ap = ap1;
  bp = bp1;
  aq = 0.0;
  if constexpr (k < 1) aq = tu[k + 2];
  y = bk;
  z = zk;
}

// One implicit-shift QR sweep over all three columns (svd.rs:495-602).
template <int R>
__device__ __forceinline__ void qr_cols3(SvdT<R>& S, double tu[3], double tv[2]) {
  if (tu[0] == 0.0) {
    qr_middle<0>(S, tu, tv);
    return;
  }
  if (tu[1] == 0.0) {
    qr_middle<1>(S, tu, tv);
    return;
  }
  if (tu[2] == 0.0) {
    qr_end(S, tu, tv);
    return;
  }
  const double mu = qr_shift(tu, tv);
  double y = tu[0] * tu[0] - mu;
  double z = tu[0] * tv[0];
  double ak = 0.0, bk = 0.0, zk = 0.0;
  double ap = tu[0], bp = tv[0], aq = tu[1];
  qr_column<0>(S, tu, tv, y, z, ak, bk, zk, ap, bp, aq);
  qr_column<1>(S, tu, tv, y, z, ak, bk, zk, ap, bp, aq);
  tv[1] = bk;
  tu[2] = ap;
}

// Diagonalisation (svd.rs:413-479).  The reference has no iteration cap;
// `max_sweeps` bounds the loop on the device so that every thread finishes
// (a cell that hits it is reported through *stalled).  The window is the last
// run of nonzero off-diagonal entries; one that has become zero at the end
// stays so.
template <int R>
__device__ __forceinline__ void diagonalise(SvdT<R>& S, double tu[3], double tv[2], int max_sweeps,
                                            bool* stalled) {
  chop<0, 3>(tu, tv);
  for (int sweeps = 0; tv[0] != 0.0 || tv[1] != 0.0; ++sweeps) {
    if (sweeps >= max_sweeps) {
      *stalled = true;
      return;
    }
    if (tv[1] == 0.0) {
      qr_cols2<0>(S, tu, tv);
      chop<0, 2>(tu, tv);
    } else if (tv[0] == 0.0) {
      qr_cols2<1>(S, tu, tv);
      chop<1, 2>(tu, tv);
    } else {
      qr_cols3(S, tu, tv);
      chop<0, 3>(tu, tv);
    }
  }
}

// Puts the greatest of the singular values from i on first (svd.rs:867-926).
template <int i, int R>
__device__ __forceinline__ void sort_column(SvdT<R>& S) {
  double dmax = S.d[i];
  int imax = i;
#pragma unroll
  for (int j = i + 1; j < 3; ++j) {
    if (S.d[j] > dmax) {
      dmax = S.d[j];
      imax = j;
    }
  }
  auto exchange = [&](auto to) {
    constexpr int j = decltype(to)::value;
    const double t = S.d[i];
    S.d[i] = S.d[j];
    S.d[j] = t;
    swap_cols<i, j, R>(S.u, S.rows);
    swap_cols<i, j, 3>(S.v, 3);
  };
  if constexpr (i == 0) {
    if (imax == 1) exchange(std::integral_constant<int, 1>{});
  }
  if (imax == 2) exchange(std::integral_constant<int, 2>{});
}

template <int R>
__device__ __forceinline__ void sort_singular(SvdT<R>& S) {
#pragma unroll
  for (int j = 0; j < 3; ++j) {
    if (S.d[j] < 0.0) {
#pragma unroll
      for (int i = 0; i < 3; ++i) S.v[i][j] = -S.v[i][j];
      S.d[j] = -S.d[j];
    }
  }
  sort_column<0>(S);
  sort_column<1>(S);
}

// TangentPlanes::new (feature/mod.rs:91-148) over n <= R points and normals
// + MinimiseQEF::place_feature_with_tangents (qef.rs:36-68); *feature
// receives whether the planes were classified Edge or Corner.
// kFull: n is R (the loops over the points are then unrolled, too).
template <int R, bool kFull>
__device__ __forceinline__ Vec3f place_feature_n(const Vec3f* corners, const Vec3f* normals,
                                                 int n, bool* stalled, bool* feature) {
  const float kFeatureAngle = 0.866025388f;  // f32(0.8660254037844387), mod.rs:22
  constexpr int kUnroll = kFull ? R : 1;
  if (kFull) n = R;
  Vec3f com{0.0f, 0.0f, 0.0f};
  int first = 0, second = 0;
  float min_angle = 3.40282347e+38f;
  float count = 0.0f;
  *feature = false;
#pragma unroll kUnroll
  for (int i = 0; i < n; ++i) {
    // (j < i repeats the angle of an earlier pair, which is not below itself)
#pragma unroll kUnroll
    for (int j = i; j < n; ++j) {
      const float angle = dot3(normals[i], normals[j]);
      if (angle < min_angle) {
        first = i;
        second = j;
        min_angle = angle;
      }
    }
    com.x += corners[i].x;
    com.y += corners[i].y;
    com.z += corners[i].z;
    count += 1.0f;
  }
  com.x /= count;
  com.y /= count;
  com.z /= count;
  if (min_angle > kFeatureAngle) return com;  // planar
  *feature = true;
  Vec3f na{0.0f, 0.0f, 0.0f}, nb{0.0f, 0.0f, 0.0f};
  if (kFull) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i == first) na = normals[i];
      if (i == second) nb = normals[i];
    }
  } else {
    na = normals[first];
    nb = normals[second];
  }
  const Vec3f axis = normalised_or_zero(cross3(na, nb));
  float min_c = 1.0f, max_c = -1.0f;
#pragma unroll kUnroll
  for (int i = 0; i < n; ++i) {
    const float c = dot3(axis, normals[i]);
    min_c = fminf(min_c, c);
    max_c = fmaxf(max_c, c);
  }
  float c = fmaxf(__builtin_fabsf(min_c), __builtin_fabsf(max_c));
  c = __builtin_sqrtf(1.0f - c * c);
  const bool edge = c > kFeatureAngle;

  SvdT<R> S;
  S.rows = n;
  double b[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    S.u[i][0] = S.u[i][1] = S.u[i][2] = b[i] = 0.0;
    if (i >= n) continue;
    S.u[i][0] = normals[i].x;
    S.u[i][1] = normals[i].y;
    S.u[i][2] = normals[i].z;
    const Vec3f r{corners[i].x - com.x, corners[i].y - com.y, corners[i].z - com.z};
    b[i] = static_cast<double>(dot3(r, normals[i]));
  }
  double tau_v[2] = {0.0, 0.0};
  bidiagonalise<R>(S.u, S.d, tau_v, n);
  unpack<R>(S.u, S.v, S.d, tau_v, n);
  diagonalise(S, S.d, tau_v, 1000, stalled);
  sort_singular(S);
  if (edge) {  // qef.rs:51-63: drop the smallest singular value
    double smin = 1.7976931348623157e308;
    int id = 0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      if (S.d[i] < smin) {
        smin = S.d[i];
        id = i;
      }
    }
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (i == id) S.d[i] = 0.0;
  }
  // SVD::solve (svd.rs:55-84) + solveSVD (svd.rs:928-972)
  if (S.d[2] < 0.1) S.d[2] = 0.0;
  if (S.d[1] < 0.1) S.d[1] = 0.0;
  if (S.d[0] < 0.1) S.d[0] = 0.0;
  double w[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int i = 0; i < R; ++i)
    if (i < n && b[i] != 0.0)
#pragma unroll
      for (int j = 0; j < 3; ++j) w[j] += b[i] * S.u[i][j];
#pragma unroll
  for (int i = 0; i < 3; ++i)
    if (S.d[i] != 0.0) w[i] /= S.d[i];
  float x[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    double t = 0.0;
#pragma unroll
    for (int j = 0; j < 3; ++j) t += w[j] * S.v[i][j];
    x[i] = static_cast<float>(t);
  }
  return {com.x + x[0], com.y + x[1], com.z + x[2]};
}

// The dual-contouring form: the 8 cell corners.
__device__ __forceinline__ Vec3f place_feature(const Vec3f corners[8], const Vec3f normals[8],
                                               bool* stalled) {
  bool feature;
  return place_feature_n<kRows, true>(corners, normals, kRows, stalled, &feature);
}

}  // namespace qef
}  // namespace iso
