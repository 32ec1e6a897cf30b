// chol16.h -- Cholesky and inverse of a 16 x 16 block in the registers of a
// 16-lane row, shared by the blocked factorisation of qr.hip and the batched one
// (batched.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace rsvd {

// v of lane J of the 16-lane row the lane is in (a data-parallel move).
template <int J>
static __device__ __forceinline__ double row_bcast(double v) {
  union {
    double d;
    int i[2];
  } u = {v};
  u.i[0] = __builtin_amdgcn_mov_dpp(u.i[0], 0x150 + J, 0xf, 0xf, true);  // row_newbcast:J
  u.i[1] = __builtin_amdgcn_mov_dpp(u.i[1], 0x150 + J, 0xf, 0xf, true);
  return u.d;
}

// Cholesky and inverse of a 16 x 16 block in the registers of a 16-lane row:
// lane c holds column c of the symmetric block (a[r], all rows) and column c of
// the identity (e[r]); step j scales row j by 1 / sqrt(pivot) and subtracts it
// from the rows below, u_jr broadcast from lane r.  On exit a[r] (r <= c) is
// R(r, c), e[r] is R^-1(c, r) (zero for r < c) and piv lane c's pivot.  The steps
// from kb on (padding) are left out.  A pivot that is not positive (or
// NaN) is replaced by 1 with FIX; without it, it gives NaN from there on.  The
// caller's test of piv reports it.
template <int J, bool FIX>
static __device__ __forceinline__ void chol16_step(double (&a)[16], double (&e)[16], int c, int kb,
                                               double* piv) {
  if (J >= kb) return;
  double d = row_bcast<J>(a[J]);
  *piv = (c == J) ? d : *piv;
  if (FIX && !(d > 0.0)) d = 1.0;
  // 1 / sqrt(d): the hardware estimate and one third-order step
  const double y0 = __builtin_amdgcn_rsq(d);
  const double r = fma(-d * y0, y0, 1.0);
  const double y = fma(y0 * r, fma(0.375, r, 0.5), y0);
  a[J] *= y;
  e[J] *= y;
  const double u = a[J], w = e[J];
  // (one compile-time broadcast a row below)
#define RSVD_CI_ROW(R)                     \
  if constexpr (R > J && R < 16) {         \
    const double m = row_bcast<R>(u);       \
    a[R] = fma(-m, u, a[R]);               \
    e[R] = fma(-m, w, e[R]);               \
  }
  RSVD_CI_ROW(1) RSVD_CI_ROW(2) RSVD_CI_ROW(3) RSVD_CI_ROW(4) RSVD_CI_ROW(5)
  RSVD_CI_ROW(6) RSVD_CI_ROW(7) RSVD_CI_ROW(8) RSVD_CI_ROW(9) RSVD_CI_ROW(10)
  RSVD_CI_ROW(11) RSVD_CI_ROW(12) RSVD_CI_ROW(13) RSVD_CI_ROW(14) RSVD_CI_ROW(15)
#undef RSVD_CI_ROW
  if constexpr (J < 15) chol16_step<J + 1, FIX>(a, e, c, kb, piv);
}

}  // namespace rsvd
