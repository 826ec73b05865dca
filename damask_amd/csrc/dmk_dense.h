// Register-resident dense solves for the per-cell Newton systems (row-major
// n x n, all indices compile-time so the matrix stays in VGPRs).
//
// The reference solves its 9x9 systems with LAPACK dgesv (LU with partial
// pivoting, src/math.f90:538-555 via src/phase_mechanical.f90:468-476,
// 1199-1208).  Row interchanges with a per-lane pivot index cannot address
// registers directly: every swap becomes a chain of selects, which costs
// several times the elimination itself on a 64-wide wavefront.  Householder
// QR needs no pivoting, is backward stable for any non-singular matrix and
// gives the same solution to rounding; that is what is used here.
//
// Singularity: a column whose remaining part is exactly zero makes R
// singular; the factorisation then reports failure, as dgesv reports info > 0
// for an exactly zero pivot.
#pragma once

#include <hip/hip_runtime.h>

#define DMK_DENSE __device__ __forceinline__

// 1/x and 1/sqrt(x): the hardware approximation and two Newton steps each
// (within 1 and 2 ulp for normal arguments and results; 0, infinity and NaN give
// NaN), without the scaling and fix-up sequences of a division and a square
// root.  The callers' arguments are positive finite state values, resolved
// stresses of a non-zero rate, and norms of non-zero columns.  An n = 5 factorisation has 5 of
// each in one dependent chain.
DMK_DENSE double dmk_rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.0), r, r);
  return fma(fma(-x, r, 1.0), r, r);
}

DMK_DENSE double dmk_rsq(double x) {
  double y = __builtin_amdgcn_rsq(x);
  const double h = 0.5 * x;
  y = fma(y, fma(-h * y, y, 0.5), y);
  return fma(y, fma(-h * y, y, 0.5), y);
}

// Factorisation J = Q R in place: R in the upper triangle without its diagonal,
// reflector tails below it; per column k the inverse diagonal of R in rd and
// the reflector I - tau v v^T with v = (v0, tail).  Returns true when J is
// singular.
template <int n>
DMK_DENSE bool dmk_qr_factor(double* J, double* rd, double* v0, double* tau) {
  bool sing = false;
#pragma unroll
  for (int k = 0; k < n; k++) {
    const double alpha = J[n * k + k];
    double s2 = alpha * alpha;
#pragma unroll
    for (int i = k + 1; i < n; i++) s2 = fma(J[n * i + k], J[n * i + k], s2);
    sing |= !(s2 > 0.0);
    const double rn = dmk_rsq(s2), nrm = s2 * rn;
    // beta = -sign(alpha) |column|, v0 = alpha - beta (no cancellation),
    // tau = 2 / (v^T v) = -1 / (beta v0)
    const double av = fabs(alpha) + nrm;
    v0[k] = copysign(av, alpha);
    tau[k] = rn * dmk_rcp(av);
    rd[k] = -copysign(rn, alpha);
#pragma unroll
    for (int j = k + 1; j < n; j++) {
      double w = v0[k] * J[n * k + j];
#pragma unroll
      for (int i = k + 1; i < n; i++) w = fma(J[n * i + k], J[n * i + j], w);
      const double s = tau[k] * w;
      J[n * k + j] = fma(-s, v0[k], J[n * k + j]);
#pragma unroll
      for (int i = k + 1; i < n; i++) J[n * i + j] = fma(-s, J[n * i + k], J[n * i + j]);
    }
  }
  return sing;
}

// J x = b for a factorised J, x returned in b
template <int n>
DMK_DENSE void dmk_qr_apply_solve(const double* J, const double* rd, const double* v0, const double* tau, double* b) {
#pragma unroll
  for (int k = 0; k < n; k++) {
    double w = v0[k] * b[k];
#pragma unroll
    for (int i = k + 1; i < n; i++) w = fma(J[n * i + k], b[i], w);
    const double s = tau[k] * w;
    b[k] = fma(-s, v0[k], b[k]);
#pragma unroll
    for (int i = k + 1; i < n; i++) b[i] = fma(-s, J[n * i + k], b[i]);
  }
#pragma unroll
  for (int k = n - 1; k >= 0; k--) {
    double s = b[k];
#pragma unroll
    for (int j = k + 1; j < n; j++) s = fma(-J[n * k + j], b[j], s);
    b[k] = s * rd[k];
  }
}
