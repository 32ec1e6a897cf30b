// jacobi_rot.h -- the 2x2 symmetric Jacobi rotation shared by the device
// eigensolvers (symeig.hip, batched.hip).
#pragma once
#include <cmath>

#include <hip/hip_runtime.h>

namespace rsvd {

// no rotation below this relative size of the off-diagonal
constexpr double kRotTol = 1e-15;
// a sweep that met no off-diagonal above this relative size ends the iteration
constexpr double kStopTol = 1e-10;
// the same for callers that need eigenvectors to fp32 level only, on the
// rotation sines |s| rather than the off-diagonal ratio: near convergence a
// pair with relative eigenvalue gap d and ratio r turns by |s| ~ r / d, and
// the next sweep leaves ratios ~ r^2 / d = s^2 d.  A sweep whose rotations
// all had |s| <= 1e-4 therefore leaves off-diagonals below ~1e-8 of
// sqrt(g_pp g_qq) for every gap (a ratio test of 1e-4 alone could stop with
// ratios of 1e-4 inside a cluster of nearly equal eigenvalues, i.e.
// first-order eigenvalue errors of 1e-4 there).  A rotation of ratio at most
// kLooseRatioTol does not count, however large its angle: inside a cluster
// (gap below 1e-4) the angles stay large until the splitting the cluster's
// members carry -- for a plateau of equal singular values, the rounding of
// the preceding stages -- is resolved to rounding, while such a pair already
// perturbs its eigenvalues by at most 1e-8 relative and leaves the columns
// of B^T V Sigma^-1 orthogonal to 1e-8.  Either way the eigenvalues are good
// to ~1e-8 relative or better and the eigenvectors of separated eigenvalues,
// and the orthogonality of B^T V Sigma^-1, to ~1e-8, below the fp32
// resolution of the outputs.
constexpr double kLooseStopTol = 1e-4;
constexpr double kLooseRatioTol = 1e-8;

// 1/x from the hardware estimate plus two Newton steps (error a few ulp).
static __device__ __forceinline__ double rcp_nr(double x) {
  double y = __builtin_amdgcn_rcp(x);
  double e = fma(-x, y, 1.0);
  y = fma(y, e, y);
  e = fma(-x, y, 1.0);
  return fma(y, e, y);
}
// The power of two that brings x > 0 to [1/2, 1); 1 for zero, NaN and Inf.
static __device__ __forceinline__ double unit_scale(double x) {
  if (!(x > 0.0) || isinf(x)) return 1.0;
  int e;
  (void)frexp(x, &e);
  // a power of two beyond the largest double is not needed: 2^-1022 times
  // 2^1022 is of order one already
  return ldexp(1.0, -e > 1022 ? 1022 : -e);
}

// The same from a squared Frobenius norm, and 0 when the square left the range
// in which it tells (the caller then scales by the largest entry).
static __device__ __forceinline__ double norm_scale(double fro2) {
  return (fro2 > 1e-280 && fro2 < 1e280) ? unit_scale(sqrt(fro2)) : 0.0;
}

// Which rotations keep the iteration going (see kStopTol, kLooseStopTol): those
// with |g| > ratio sqrt|ab| and |t| > angle.
struct RotStop {
  float ratio2, angle;
};
static __host__ __device__ __forceinline__ RotStop rot_stop(bool loose) {
  return loose ? RotStop{(float)(kLooseRatioTol * kLooseRatioTol), (float)kLooseStopTol}
               : RotStop{(float)(kStopTol * kStopTol), -1.0f};
}

// Rotation (c, s) with [x' y'] = [x y] [[c, s], [-s, c]] zeroing the (p, q)
// entry of a symmetric 2x2 [[a, g], [g, b]] of a matrix scaled to norm 1
// (unit_scale): t = tan theta is the root of g t^2 + (b - a) t - g = 0 of
// smaller modulus, t = sgn(d) 2g / (|d| + r), d = b - a, r = sqrt(d^2 + 4g^2)
// (Rutishauser's choice).  The angle only has to be close: t is formed in
// single precision (relative error below 1e-6, so a rotation leaves less than
// 1e-6 of its off-diagonal, which the caller's update computes like any other
// entry); everything above flo (1e-15 of the norm) keeps its square in range.
// That (c, s) is a rotation to rounding is what orthogonality rests on:
// c = 1 / sqrt(1 + t^2) in double precision from the single precision estimate
// and one third-order step (error below 1e-20 before rounding), s = c t.
// Measured, largest eigenvalue error over the norm, random symmetric matrices of
// n = 20 / 110 / 200: 1.8e-15 / 9.0e-15 / 2.0e-14 with the angle formed in double
// precision, 0.95e-15 / 5.0e-15 / 0.8e-14 with this one (fewer roundings in c and s);
// residual and orthogonality are smaller too.
// Branch-free.  No rotation when |g| <= flo or |g| <= kRotTol sqrt|ab|; *sig
// tells whether the rotation counts for `stop`.
// What bounds a rotation step is the issue of its instructions (a wave issues
// one every four cycles and has its SIMD to itself): this form has 35, two
// reciprocal square roots in double precision with two Newton steps each, the
// scaling of each triple and the tests in double precision had about 80.
static __device__ __forceinline__ void rotation(double a, double b, double g, float flo,
                                                RotStop stop, double* cs, double* sn, bool* sig) {
  const double d = b - a;
  const float af = (float)a, bf = (float)b, gf = (float)g, df = (float)d;
  const float ab = fabsf(af * bf), g2 = gf * gf;
  const float r = __builtin_amdgcn_sqrtf(fmaf(df, df, 4.0f * g2));
  const float q = (gf + gf) * __builtin_amdgcn_rcpf(fabsf(df) + r);
  const bool rot = (fabsf(gf) > flo) & (g2 > (float)(kRotTol * kRotTol) * ab);
  const float t = rot ? copysignf(1.0f, df) * q : 0.0f;
  const double td = (double)t, x = fma(td, td, 1.0);
  const double y = (double)__builtin_amdgcn_rsqf(fmaf(t, t, 1.0f));
  const double e = fma(-x * y, y, 1.0);
  const double c = fma(y * e, fma(0.375, e, 0.5), y);
  *cs = c;
  *sn = c * td;
  *sig = rot & (g2 > stop.ratio2 * ab) & (fabsf(t) > stop.angle);
}

}  // namespace rsvd
