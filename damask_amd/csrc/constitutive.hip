// Per-material-point constitutive update on MI355X: one lane per cell, FP64.
//
// stress_kernel: homogenization_mechanical_response's first loop
//   (src/homogenization.f90:309-348): restore, isostrain partition,
//   phase_mechanical_constitutive substepping (src/phase_mechanical.f90:1008-1090),
//   integrateStateFPI (:591-676) and integrateStress (:379-584) with
//   phenopowerlaw kinetics (src/phase_mechanical_plastic_phenopowerlaw.f90:303-399,449-488)
//   and Hooke's law (src/phase_mechanical_elastic.f90:172-205).
// tangent_kernel: the second loop (:352-360): crystallite orientation
//   (src/phase.f90:659-673) and phase_mechanical_dPdF (src/phase_mechanical.f90:1121-1242).
//
// The material point carries no eigen kinematics and V_e = I, so F_i = I and
// L_i = 0 throughout; the 3x3x3x3 chains of the reference then collapse to
// rank-N_sl updates of the 9x9 identity:
//   dR_Lp/dL_p = I9 + dt * sum_a dgamma_a vec(P_a) vec(G^T Q_a)^T,  G = F_e^T A,
//   Q_a = C : P_nS,a,
// whose rank is at most that of the symmetric tensors the Q_a span, 5 with the
// Schmid law and 6 with non-Schmid terms: the Newton step and the consistent
// tangent are solved in that space (integrate_stress, tangent_kernel), by
// Householder QR in registers (dmk_dense.h).
//
// What bounds the stress kernel: FP64 issue and the latency of a wavefront's own
// chain (Newton steps in sequence, each with a QR and scalar table loads), not
// HBM.  64^3 cells of the cF tension, 5.5 Newton iterations a cell: 0.286 ms a
// launch, 0.69 ms as an 8x8 system per Newton step with the state in global
// scratch; 45x50x54 cells with 24 systems 0.36 against 0.95 ms; 16^3 cells (one
// wavefront a CU) 0.09 against 0.21 ms.
// Register budget: between the Newton steps only A and L_p live in registers;
// per-system values (1/xi, d rate / d tau, rates), the Newton direction and the
// sub-step bookkeeping live in LDS, [system][lane], one wavefront per
// work-group; the state-rate history of the fixed-point iteration is in global
// scratch.
#include <cmath>

#include "dmk_common.h"
#include "dmk_math.h"
#include "dmk_dense.h"

namespace {

constexpr int SWG = DMK_STRESS_WG;   // work-group of the per-cell kernels: one wavefront

// Wavefronts per SIMD.  12 systems: two (256 registers, a few spills) hide each
// other's latency: 0.275 ms a launch at 64^3 against 0.36 ms with one and no
// spills.  24 systems: the LDS vectors leave room for five work-groups a CU and
// the state update holds 144 values, so one (512 registers): 0.36 ms at
// 45x50x54 against 0.66 ms with two; non-Schmid terms alike (0.59 against 1.17 ms
// at 48^3 with half the cells in such a phase).
constexpr int stress_waves(int nsl) { return nsl > 12 ? 1 : 2; }

// Library transcendental functions are kept out of line: inlined, their
// polynomial constants are hoisted out of every enclosing loop and stay live
// across the 9x9 Newton system.
__device__ __noinline__ double pow_ool(double x, double y) { return pow(x, y); }
// four at once: their chains overlap (31x45x27 cells, 24 systems, n = 17.3: 0.412
// instead of 0.477 ms a launch; 64^3 cells, 12 systems 0.595 instead of 0.631)
struct Four { double v[4]; };
__device__ __noinline__ Four pow4_ool(Four x, Four y) {
#pragma unroll
  for (int j = 0; j < 4; j++) x.v[j] = pow(x.v[j], y.v[j]);
  return x;
}
__device__ __noinline__ double tanh_ool(double x) { return tanh(x); }

// x^y for the power laws (phenopowerlaw n_sl, a_sl).  With QP (every
// exponent of the phase is a positive multiple of 1/4 up to 64, checked on the
// host) y = k/4 is evaluated by binary powering of x (k a multiple of 4),
// sqrt(x) (k even) or sqrt(sqrt(x)) (k odd); y is a per-phase constant, so the
// powering loop is uniform across the wavefront.  Its error is that of the
// root, amplified by the power taken of it, plus the products' roundings,
// each amplified by the powering after it; against a long-double reference
// over the power laws' base ranges: n = 20 within 12 ulp, a = 2.25 within 11
// ulp, a = 2 within 0.5 ulp, and up to 376 ulp (8e-14 relative) for the
// largest odd multiples of 1/4 (y near 64, taken as (x^(1/4))^255).  It
// follows pow's rules for zero, negative (NaN unless y is an integer, sign of
// odd powers), infinite and NaN bases.  Phases with other exponents use the
// library pow (within 2 ulp), four systems at a time (pow_laws).
template <bool QP>
DI double pow_law(double x, double y) {
  if (!QP) return pow_ool(x, y);
  int k = (int)(y * 4.0);
  double b = x;
  if (k & 1) {
    b = sqrt(sqrt(x));
  } else if (k & 2) {
    b = sqrt(x);
    k >>= 1;
  } else {
    k >>= 2;
  }
  double r = 1.0;
  bool first = true;
  while (k) {
    if (k & 1) { r = first ? b : r * b; first = false; }
    k >>= 1;
    if (k) b = b * b;
  }
  return r;
}

// xs_a <- xs_a^y_a of systems a0 .. a0 + n - 1 (LDS), n a multiple of 4
template <bool QP, class Table>
DI void pow_laws(Table y, int a0, int n, double* xs) {
  if (QP) {
#pragma unroll 1
    for (int j = a0; j < a0 + n; j++) xs[j * SWG] = pow_law<QP>(xs[j * SWG], y[j]);
  } else {
#pragma unroll 1
    for (int j = a0; j < a0 + n; j += 4) {
      Four x, e;
#pragma unroll
      for (int k = 0; k < 4; k++) { x.v[k] = xs[(j + k) * SWG]; e.v[k] = y[j + k]; }
      x = pow4_ool(x, e);
#pragma unroll
      for (int k = 0; k < 4; k++) xs[(j + k) * SWG] = x.v[k];
    }
  }
}

// the power laws' x^y on the device, for checking their arithmetic
template <bool QP>
__global__ void pow_law_kernel(const double* __restrict__ x, const double* __restrict__ y, double* __restrict__ out,
                               int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = pow_law<QP>(x[i], y[i]);
}

// Coordinates of the per-cell algebra.  The Schmid tensors are traceless, and
// with them every plastic quantity lies in the span of eight constant tensors:
// five symmetric deviators E_1 = diag(1,-1,0)/sqrt2, E_2 = diag(1,1,-2)/sqrt6,
// E_3..E_5 = (e_i e_j + e_j e_i)/sqrt2 for (ij) = (12), (02), (01), and three
// skew ones R_m = (e_i e_j - e_j e_i)/sqrt2 for the same pairs, an orthonormal
// set.  Cubic elasticity is diagonal in E (C11 - C12, C11 - C12, 2 C44 x 3), and
// a resolved stress is S : P_nS_a with S symmetric, so of the projections only
// the E part acts: 5 numbers per system, with non-Schmid terms 6
// (E_6 = I/sqrt3, modulus C11 + 2 C12).  Per phase: sp = (E, R) of P_a, qp / qm =
// E of P_nS_a in the positive / negative sense.
constexpr double R2 = 0.70710678118654752440;   // 1/sqrt2
constexpr double R3 = 0.57735026918962576451;   // 1/sqrt3
constexpr double R6 = 0.40824829046386301637;   // 1/sqrt6

// The phase tables are read through the constant address space: the addresses
// are uniform, so every read is a scalar load.  Through a plain pointer the
// compiler takes vector loads in loops that also store, 2000 a wavefront, each a
// trip to L2 in the Newton's dependency chain (0.53 instead of 0.35 ms at 64^3
// when this was measured alone).
using PhPtr = const __attribute__((address_space(4))) DmkPhaseDev*;

template <bool NS>
constexpr int sym_rank() { return NS ? 6 : 5; }

// E_k : X of any 3x3
template <int RK>
DI void sym_proj(const double* X, double* t) {
  t[0] = (X[0] - X[4]) * R2;
  t[1] = (X[0] + X[4] - 2.0 * X[8]) * R6;
  t[2] = (X[5] + X[7]) * R2;
  t[3] = (X[2] + X[6]) * R2;
  t[4] = (X[1] + X[3]) * R2;
  if (RK == 6) t[5] = (X[0] + X[4] + X[8]) * R3;
}

// sum_k h_k E_k + sum_m k_m R_m
DI void from_basis(const double* h, const double* k, double* X) {
  const double a = h[0] * R2, b = h[1] * R6;
  X[0] = b + a;
  X[4] = b - a;
  X[8] = -2.0 * b;
  double s = h[2] * R2, q = k[0] * R2;
  X[5] = s + q; X[7] = s - q;
  s = h[3] * R2; q = k[1] * R2;
  X[2] = s + q; X[6] = s - q;
  s = h[4] * R2; q = k[2] * R2;
  X[1] = s + q; X[3] = s - q;
}

// modulus of E_k
template <int RK>
DI double modulus(PhPtr ph, int k) {
  return k < 2 ? ph->C11 - ph->C12 : (k < 5 ? 2.0 * ph->C44 : ph->C11 + 2.0 * ph->C12);
}

// E_k : S of S = C : (Fe^T Fe - I)/2.  The diagonal sums start at -1, so that
// their roundings are those of the small strain's last steps.
template <int RK>
DI void stress_coords(PhPtr ph, const double* Fe, double* s) {
  double c[6];   // Fe^T Fe - I: 00, 11, 22, 12, 02, 01
#pragma unroll
  for (int q = 0; q < 6; q++) {
    const int i = q < 3 ? q : (q == 3 ? 1 : 0), j = q < 3 ? q : (q == 5 ? 1 : 2);
    double v = q < 3 ? fma(Fe[i], Fe[j], -1.0) : Fe[i] * Fe[j];
    v = fma(Fe[3 + i], Fe[3 + j], v);
    c[q] = fma(Fe[6 + i], Fe[6 + j], v);
  }
  const double d = 0.5 * (ph->C11 - ph->C12), g = ph->C44;
  s[0] = (c[0] - c[1]) * (d * R2);
  s[1] = (c[0] + c[1] - 2.0 * c[2]) * (d * R6);
  s[2] = c[3] * (2.0 * R2 * g);
  s[3] = c[4] * (2.0 * R2 * g);
  s[4] = c[5] * (2.0 * R2 * g);
  if (RK == 6) s[5] = (c[0] + c[1] + c[2]) * (0.5 * R3 * (ph->C11 + 2.0 * ph->C12));
}

// per-lane slip-system vectors, entry a of a lane at [a][lane]
template <int NSL>
struct SlipLds {
  double g[NSL][SWG];     // d rate / d tau in the stress Newton loop, |rate| in the state loop
  double w[NSL][SWG];     // 1 / xi in the stress Newton loop, xi rate in the state loop
  double dir[9][SWG];     // the Newton direction, read back when a step is rejected
  // sub-step bookkeeping of a lane, kept out of the registers the Newton needs
  double frac[SWG], step[SWG];
  int nsub[SWG], fpi[SWG];
};

// The slip-system loops take CH systems at once, so that their chains overlap,
// and read the phase tables in batches of GRP systems (64 scalar registers);
// batch_end keeps the compiler from loading the batches all together, which are
// more values than there are scalar registers.  What a loop leaves for another
// goes through LDS, [system][lane].
constexpr int CH = 12, GRP = 4;

DI void batch_end() { __builtin_amdgcn_sched_barrier(0); }

// resolved stress of system a: signed tau with the Schmid law, max(tau+, tau-)
// with non-Schmid terms (pos: the positive sense acts)
template <bool NS>
DI double resolved(PhPtr ph, int a, const double* s, bool& pos) {
  // the Schmid law projects on P itself
  double tp = s[0] * (NS ? ph->qp[a][0] : ph->sp[a][0]);
#pragma unroll
  for (int k = 1; k < sym_rank<NS>(); k++) tp = fma(s[k], NS ? ph->qp[a][k] : ph->sp[a][k], tp);
  if (!NS) {
    pos = tp > 0.0;
    return tp;
  }
  double tn = s[0] * ph->qm[a][0];
#pragma unroll
  for (int k = 1; k < sym_rank<NS>(); k++) tn = fma(s[k], ph->qm[a][k], tn);
  pos = tp > tn;
  return fmax(tp, tn);
}

// x_j^(k/4) of n values with one binary powering of x, sqrt(x) or sqrt(sqrt(x)),
// as pow_law takes one: the branches are taken once and the products are n
// independent chains.  Largest errors against long double: the rates' x^(n-1) x
// 10.7 ulp at n = 20 (pow_law: 12) and 115 at n = 20.25, the hardening's x^a 11 at
// a = 2.25 and 0.5 at a = 2.
template <int n>
DI void quarter_power(double* x, int k) {
  if (k & 3) {
#pragma unroll
    for (int j = 0; j < n; j++) x[j] = sqrt(x[j]);
    if (k & 1) {
#pragma unroll
      for (int j = 0; j < n; j++) x[j] = sqrt(x[j]);
    } else {
      k >>= 1;
    }
  } else {
    k >>= 2;
  }
  double r[n];
#pragma unroll
  for (int j = 0; j < n; j++) r[j] = 1.0;
  while (k) {
    if (k & 1) {
#pragma unroll
      for (int j = 0; j < n; j++) r[j] *= x[j];
    }
    k >>= 1;
    if (k) {
#pragma unroll
      for (int j = 0; j < n; j++) x[j] *= x[j];
    }
  }
#pragma unroll
  for (int j = 0; j < n; j++) x[j] = r[j];
}

// kinetics_sl (src/phase_mechanical_plastic_phenopowerlaw.f90:449-488) of all
// systems of one lane at the stress coordinates s; ixs: 1/xi per system (LDS).
// NEWTON: gs <- d rate / d tau (0 where the rate is 0), L_p = sum_a rate_a P_a in
// basis coordinates l (E) and k3 (R), posm: bit a set where the positive sense
// of system a acts; otherwise gs <- |rate|.
// A phase whose systems share one exponent n >= 1, a multiple of 1/4 (n_k = 4 n),
// takes x^(n-1) of CH systems by one powering, then x^n = x^(n-1) x and
// n x^(n-1) / xi without a division; others take one power after the other
// (rolled: the out-of-line pow then has one call site).
template <int NSL, bool QP, bool NS, bool NEWTON>
DI void kinetics(PhPtr ph, const double* s, const double* ixs, double* gs, double* l,
                 double* k3, unsigned& posm) {
  if (NEWTON) {
#pragma unroll
    for (int k = 0; k < 5; k++) l[k] = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++) k3[m] = 0.0;
    posm = 0;
  }
  const int nk = QP ? ph->n_k : 0;
#pragma unroll 1
  for (int a0 = 0; a0 < NSL; a0 += CH) {
    double x[CH], r[CH];
    unsigned pm = 0;
#pragma unroll
    for (int j = 0; j < CH; j++) {
      bool pos;
      x[j] = resolved<NS>(ph, a0 + j, s, pos) * ixs[(a0 + j) * SWG];
      if (NS && pos) pm |= 1u << j;
      if (j % GRP == GRP - 1) batch_end();
    }
    if (NEWTON) posm |= pm << a0;
    if (QP && nk) {
#pragma unroll
      for (int j = 0; j < CH; j++) r[j] = NS ? x[j] : fabs(x[j]);
      quarter_power<CH>(r, nk - 4);                    // x^(n-1)
    } else {
#pragma unroll
      for (int j = 0; j < CH; j++) gs[(a0 + j) * SWG] = NS ? x[j] : fabs(x[j]);
      pow_laws<QP>(&ph->n[0], a0, CH, gs);
#pragma unroll
      for (int j = 0; j < CH; j++) r[j] = gs[(a0 + j) * SWG];
    }
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const int a = a0 + j;
      const double ixi = ixs[a * SWG];
      const bool pos = NS ? (pm >> j) & 1u : x[j] > 0.0;
      double g, w;
      if (QP && nk) {
        const double f = NS && !pos ? -ph->g0[a] : ph->g0[a];
        g = f * (r[j] * x[j]);
        w = f * ph->n[a] * (r[j] * ixi);
      } else {
        g = (pos ? ph->g0[a] : -ph->g0[a]) * r[j];
        w = g * ph->n[a] * ixi * dmk_rcp(x[j]);
      }
      if (NEWTON) {
        gs[a * SWG] = !dEq0(g) ? w : 0.0;
#pragma unroll
        for (int k = 0; k < 5; k++) l[k] = fma(g, ph->sp[a][k], l[k]);
#pragma unroll
        for (int m = 0; m < 3; m++) k3[m] = fma(g, ph->sp[a][5 + m], k3[m]);
        if (j % GRP == GRP - 1) batch_end();
      } else {
        gs[a * SWG] = fabs(g);
      }
    }
  }
}

// |rate| from the derivatives that kinetics left in gs: rate = tau (d rate / d tau) / n
template <int NSL, bool NS>
DI void rates_of_derivatives(PhPtr ph, const double* s, double* gs) {
#pragma unroll 1
  for (int a0 = 0; a0 < NSL; a0 += CH) {
#pragma unroll
    for (int j = 0; j < CH; j++) {
      bool pos;
      const int a = a0 + j;
      gs[a * SWG] = fabs(gs[a * SWG] * resolved<NS>(ph, a, s, pos) * ph->inv_n[a]);
      if (j % GRP == GRP - 1) batch_end();
    }
  }
}

// W_l = sum_a u_a q_al P_a, u_a = scale * us_a (LDS), for the acting projections
// q (E coordinates): its E coordinates H[k][l] and R coordinates K[m][l].  With
// the Schmid law q = p of the same system and H is symmetric (15 products
// instead of 25).
template <int NSL, bool NS>
DI void slip_moments(PhPtr ph, const double* us, double scale, unsigned posm,
                     double (*H)[sym_rank<NS>()], double (*K)[sym_rank<NS>()]) {
  constexpr int RK = sym_rank<NS>(), G = NS ? 2 : GRP;
#pragma unroll
  for (int l = 0; l < RK; l++) {
#pragma unroll
    for (int k = 0; k < 5; k++) H[k][l] = 0.0;
#pragma unroll
    for (int m = 0; m < 3; m++) K[m][l] = 0.0;
  }
#pragma unroll 1
  for (int a0 = 0; a0 < NSL; a0 += G) {
#pragma unroll
    for (int j = 0; j < G; j++) {
      const int a = a0 + j;
      const bool pos = (posm >> a) & 1u;
      const double u = scale * us[a * SWG];
#pragma unroll
      for (int l = 0; l < RK; l++) {
        const double v = u * (NS ? (pos ? ph->qp[a][l] : ph->qm[a][l]) : ph->sp[a][l]);
#pragma unroll
        for (int k = NS ? 0 : l; k < 5; k++) H[k][l] = fma(v, ph->sp[a][k], H[k][l]);
#pragma unroll
        for (int m = 0; m < 3; m++) K[m][l] = fma(v, ph->sp[a][5 + m], K[m][l]);
      }
    }
  }
  if (!NS) {
#pragma unroll
    for (int l = 1; l < RK; l++)
#pragma unroll
      for (int k = 0; k < l; k++) H[k][l] = H[l][k];
  }
}

// The 9x9 systems of the material point (identity plus one rank-1 term per
// slip system) reduced to the RK symmetric directions: with W_l as above and
// t_k(X) = E_k : (G X), N_kl = delta_kl + C_k t_k(W_l), C_k the modulus of E_k (any
// of them may be zero).
template <int RK>
DI void reduced_matrix(PhPtr ph, const double* G, const double (*H)[RK],
                       const double (*K)[RK], double* N) {
#pragma unroll
  for (int l = 0; l < RK; l++) {
    double h[5], k3[3], W[9], GW[9], t[6];
#pragma unroll
    for (int k = 0; k < 5; k++) h[k] = H[k][l];
#pragma unroll
    for (int m = 0; m < 3; m++) k3[m] = K[m][l];
    from_basis(h, k3, W);
    m_mul(G, W, GW);
    sym_proj<RK>(GW, t);
#pragma unroll
    for (int k = 0; k < RK; k++) N[RK * k + l] = k == l ? fma(modulus<RK>(ph, k), t[k], 1.0) : modulus<RK>(ph, k) * t[k];
  }
}

// sum_l y_l W_l
template <int RK>
DI void moments_apply(const double (*H)[RK], const double (*K)[RK], const double* y, double* X) {
  double h[5], k3[3];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    h[k] = H[k][0] * y[0];
#pragma unroll
    for (int l = 1; l < RK; l++) h[k] = fma(H[k][l], y[l], h[k]);
  }
#pragma unroll
  for (int m = 0; m < 3; m++) {
    k3[m] = K[m][0] * y[0];
#pragma unroll
    for (int l = 1; l < RK; l++) k3[m] = fma(K[m][l], y[l], k3[m]);
  }
  from_basis(h, k3, X);
}

// phenopowerlaw_dotState without twins (src/phase_mechanical_plastic_phenopowerlaw.f90:356-397)
// from the gamma rates gs = |slip rate| at the state xi(r): ws <- xi rate.
// xi_sat = xi_inf + f_sat sqrt(sum F_tw) and hf = h_0 (1 + c_1 (sum F_tw)^c_2) at sum F_tw = 0
// are tabulated per phase.  Returns true when a rate is NaN.
// xi / xi_sat is the rounded quotient: xi times the rounded 1 / xi_sat, corrected
// by its residual (Markstein, IBM J. Res. Dev. 34(1) 1990), so that 1 - xi / xi_sat is
// exactly 0 where xi = xi_sat, as a power a_sl < 1 of it needs; 1 / xi in ws would
// leave 2e-16 there.  It costs the way of xi from memory: a stress launch of 64^3
// cells, 12 systems, 276 -> 286 us, of 45x50x54, 24 systems, 366 -> 363.  With the
// sums over the acting systems first, while xi is on its way, it took 287 and 370
// (hg stays in registers over the powering), with the other rows loaded ahead as well up to 335.
template <int NSL, bool QP, class State>
DI bool dot_state(PhPtr ph, State xi, const double* gs, double* ws) {
  const int ak = QP ? ph->a_k : 0;
#pragma unroll
  for (int r0 = 0; r0 < NSL; r0 += CH) {
    double x[CH], p[CH];
#pragma unroll
    for (int j = 0; j < CH; j++) {
      const double v = xi(r0 + j), inv = ph->inv_xi_sat[r0 + j], q = v * inv;
      x[j] = 1.0 - fma(fma(-q, ph->xi_sat[r0 + j], v), inv, q);
    }
    if (QP && ak) {
#pragma unroll
      for (int j = 0; j < CH; j++) p[j] = fabs(x[j]);
      quarter_power<CH>(p, ak);
    } else {
#pragma unroll
      for (int j = 0; j < CH; j++) ws[(r0 + j) * SWG] = fabs(x[j]);
      pow_laws<QP>(&ph->a[0], r0, CH, ws);
#pragma unroll
      for (int j = 0; j < CH; j++) p[j] = ws[(r0 + j) * SWG];
    }
#pragma unroll
    for (int j = 0; j < CH; j++) ws[(r0 + j) * SWG] = ph->hf[r0 + j] * copysign(p[j], x[j]);
  }
  double hg[NSL];
#pragma unroll
  for (int r = 0; r < NSL; r++) hg[r] = 0.0;
  bool nan = false;
#pragma unroll 48 / NSL
  for (int a = 0; a < NSL; a++) {
    const double ga = gs[a * SWG];
    nan |= (ga != ga);
#pragma unroll
    for (int r = 0; r < NSL; r++) hg[r] = fma(ph->Hc[a][r], ga, hg[r]);
  }
#pragma unroll
  for (int r = 0; r < NSL; r++) {
    const double d = ws[r * SWG] * hg[r];
    ws[r * SWG] = d;
    nan |= (d != d);
  }
  return nan;
}

// E = (Fe^T Fe - I)/2 and S = C:E (lattice frame)
DI void hooke(PhPtr ph, const double* Fe, double* S) {
  double E[9];
  m_mul_tn(Fe, Fe, E);
  E[0] -= 1.0; E[4] -= 1.0; E[8] -= 1.0;
#pragma unroll
  for (int k = 0; k < 9; k++) E[k] *= 0.5;
  hooke_sym(ph->C11, ph->C12, ph->C44, E, S);
}

// The material-point arguments are read through the constant address space
// too, where they are used: an argument pointer is a scalar load away, while keeping
// all of them (and the component bases formed from them) in scalar registers
// across the Newton loop spills them into vector lanes.
using MpPtr = const __attribute__((address_space(4))) DmkMPDev*;

DI MpPtr fresh(MpPtr m) {
  asm volatile("" : "+s"(m));
  return m;
}

// n rows of a field from row c on: where a sub-step has completed (started) they
// come from the sub-step scratch q, else from the increment's field f.  Almost no
// wavefront holds a started cell: the scratch is read only in those that do.
template <int n>
DI void ld_start(const double* f, const double* q, bool started, const Lane& l, int c, double* v) {
#pragma unroll
  for (int r = 0; r < n; r++) v[r] = ld(f, l, c + r);
  if (__builtin_expect(__any(started), 0)) {
#pragma unroll
    for (int r = 0; r < n; r++) {
      const double u = ld(q, l, c + r);
      v[r] = started ? u : v[r];
    }
  }
}

DI void m_load_start(const double* f, const double* q, bool started, const Lane& l, double* T) {
  m_load(f, l, T);
  if (__builtin_expect(__any(started), 0)) {
    double U[9];
    m_load(q, l, U);
#pragma unroll
    for (int k = 0; k < 9; k++) T[k] = started ? U[k] : T[k];
  }
}

// per-cell scratch of the stress integration ([DMK_SUB_ROWS][N]), written once
// a sub-step has completed: its F, F_p and L_p, where the next one starts
enum { SUB_F0 = 0, SUB_FP0 = 9, SUB_LP0 = 18 };
static_assert(SUB_LP0 + 9 <= DMK_SUB_ROWS, "sub-step scratch rows");

// F of a sub-step: its start plus step (F - F_0)
DI void sub_F(MpPtr m, const double* Ftarget, bool started, const Lane& ln, double step, double* F) {
  MpPtr q = fresh(m);
  double F0[9], Ft[9];
  m_load(q->F0, ln, F0);
  m_load(Ftarget, ln, Ft);
  m_load_start(q->F0, q->sub + SUB_F0 * ln.sN, started, ln, F);
#pragma unroll
  for (int k = 0; k < 9; k++) F[k] = fma(step, Ft[k] - F0[k], F[k]);
}

// I - dt L_p
DI void flow(double dt, const double* Lp, double* B) {
#pragma unroll
  for (int k = 0; k < 9; k++) B[k] = ((k % 4) == 0 ? 1.0 : 0.0) - dt * Lp[k];
}

// F_e = A (I - dt L_p) as A - dt (A L_p): one rounding at the size of F_e per
// entry.  The stress, and n times as much the rates, see this rounding through
// the elastic stiffness; it is the floor of the Newton iteration's residual
// (below 5e-12 of L_p: a 32^3 tension converges at that tolerance).
DI void elastic_F(double dt, const double* A, const double* Lp, double* Fe) {
  m_mul(A, Lp, Fe);
#pragma unroll
  for (int k = 0; k < 9; k++) Fe[k] = fma(-dt, Fe[k], A[k]);
}

// integrateStress (src/phase_mechanical.f90:379-584) with F_i = I, L_i = 0 for
// A = F F_p0^-1, starting from Lp, which holds the converged L_p on success.
// ixs (LDS): 1/xi per system; on success sh.g holds the |slip rates| at (S, xi).
// S, P, F_p and F_e follow from (A, F_p0, L_p) alone, so they are formed once, by
// finish_point, after the state integration has converged.
//
// The Newton system (I9 + sum_a u_a vec(P_a) vec(G^T C:P_nS_a)^T) x = res,
// G = F_e^T A, u_a = dt d rate_a / d tau_a, is the identity plus a map that sees
// x only through t_k(x) = E_k : (G x): with y_l = C_l t_l(x),
//   x = res - sum_l y_l W_l,   N y = C t(res),   N_kl = delta_kl + C_k t_k(W_l),
// W_l = sum_a u_a q_al P_a.  So a 5x5 system (6x6 with non-Schmid terms) is
// assembled and solved instead of an 8x8 one: the same Newton step.
template <int NSL, bool QP, bool NS>
DI int integrate_stress(PhPtr ph, const DmkNumMech& num, const double* A, double det_Fp0,
                        double dt, SlipLds<NSL>& sh, int lane, int& newton, double* Lp) {
  constexpr int RK = sym_rank<NS>();
  const double* ixs = &sh.w[0][lane];
  double* gs = &sh.g[0][lane];
  double* dir = &sh.dir[0][lane];
#pragma unroll
  for (int k = 0; k < 9; k++) dir[k * SWG] = 0.0;
  // norms are compared squared (a tolerance whose square underflows still takes a residual of 0)
  const double er2 = num.eps_rel_Lp * num.eps_rel_Lp, ea2 = fmax(num.eps_abs_Lp * num.eps_abs_Lp, 4.9e-324);
  double step = 1.0, res_old = DBL_MAX;
  int it = 0;
  for (;;) {
    it++;
    if (it > num.N_iter_Lp_max) return ST_FAIL_LP_MAXIT;
    newton++;
    double Fe[9], res[9];
    unsigned posm;
    {
      double s[6], l[5], k3[3], Lpc[9];
      elastic_F(dt, A, Lp, Fe);
      stress_coords<RK>(ph, Fe, s);
      kinetics<NSL, QP, NS, true>(ph, s, ixs, gs, l, k3, posm);
      from_basis(l, k3, Lpc);
      const double ng = m_norm2(Lp), nc = m_norm2(Lpc);
#pragma unroll
      for (int k = 0; k < 9; k++) res[k] = Lp[k] - Lpc[k];
      const double nres = m_norm2(res);
      if (nres != nres) return ST_FAIL_LP_NAN;
      if (nres < fmax(er2 * fmax(ng, nc), ea2)) {
        rates_of_derivatives<NSL, NS>(ph, s, gs);
        double B[9];
        flow(dt, Lp, B);
        // the reference's error exit when the new plastic deformation is singular
        // (math_invert33 of F_p0^-1 (I - dt L_p))
        return dEq0(m_det(B) / det_Fp0) ? ST_FAIL_STRESS : ST_OK;
      }
      if (!(nres < res_old)) {
        // back along the direction from the last accepted L_p
        const double back = num.r_linesearch_Lp * step - step;
        step = num.r_linesearch_Lp * step;
#pragma unroll
        for (int k = 0; k < 9; k++) Lp[k] = fma(dir[k * SWG], back, Lp[k]);
        continue;
      }
      res_old = nres;
      step = 1.0;
    }
    // Jacobian, rebuilt every iteration (f_update_jacobi_Lp = 1)
    double H[5][RK], K[3][RK], y[6];
    slip_moments<NSL, NS>(ph, gs, dt, posm, H, K);
    {
      double G[9], N[RK * RK], GX[9], rd[RK], v0[RK], tau[RK];
      m_mul_tn(Fe, A, G);
      reduced_matrix<RK>(ph, G, H, K, N);
      m_mul(G, res, GX);
      sym_proj<RK>(GX, y);
#pragma unroll
      for (int k = 0; k < RK; k++) y[k] *= modulus<RK>(ph, k);
      if (dmk_qr_factor<RK>(N, rd, v0, tau)) return ST_FAIL_LP_DGESV;
      dmk_qr_apply_solve<RK>(N, rd, v0, tau, y);
    }
    double X[9];
    moments_apply<RK>(H, K, y, X);
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const double d = X[k] - res[k];
      dir[k * SWG] = d;
      Lp[k] += d;
    }
  }
}

// The end of integrateStress (src/phase_mechanical.f90:571-581) of a sub-step:
// F_e = A (I - dt L_p) and S = C:(F_e^T F_e - I)/2; the regularised
// F_p = F_p,new / det(F_p,new)^(1/3) goes to Fp_dst; with OUT also
// P = F_e S F_p,new^-T and F_e.
template <bool OUT>
DI void finish_point(PhPtr ph, MpPtr m, const Lane& ln, bool started, const double* A,
                     const double* Lp, double dt, double* Fp_dst) {
  double invFp_new[9], Fp_new[9], Fe[9], S[9];
  {
    double Fp0[9], invFp0[9], B[9];
    MpPtr q = fresh(m);
    m_load_start(q->Fp0, q->sub + SUB_FP0 * ln.sN, started, ln, Fp0);
    m_invert(Fp0, invFp0);
    flow(dt, Lp, B);
    m_mul(invFp0, B, invFp_new);
  }
  elastic_F(dt, A, Lp, Fe);
  hooke(ph, Fe, S);
  m_store(fresh(m)->S, ln, S);
  if (OUT) {
    double T[9], P[9];
    m_mul_nt(S, invFp_new, T);
    m_mul(Fe, T, P);
    m_store(fresh(m)->Pph, ln, P);
    m_store(fresh(m)->Fe, ln, Fe);
  }
  m_invert(invFp_new, Fp_new);
  double d = pow_ool(m_det(Fp_new), 1.0 / 3.0);
#pragma unroll
  for (int k = 0; k < 9; k++) Fp_new[k] = Fp_new[k] / d;
  m_store(Fp_dst, ln, Fp_new);
}

// integrateStateFPI (src/phase_mechanical.f90:591-676).  State = (xi, gamma),
// started from xi0 / gam0 (the converged increment, or st0s after a completed
// sub-step).  Every iterate of the state is its start plus dt times the last
// damped rate: the two previous ones (dotState_last) are kept in the ping-pong
// buffers mp.last1 / mp.last2, and each iteration stores its xi and gamma.  The
// initial rate is taken at the stress S_0 after a restore, else at the previous
// sub-step's S (s_cur).  A and Lp stay in registers; on success Lp holds the converged L_p.
template <int NSL, bool QP, bool NS>
DI int integrate_state_fpi(PhPtr ph, const DmkNumMech& num, MpPtr m,
                           const double* Ftarget, const Lane& ln, bool started, bool s_cur, double step, double dt,
                           SlipLds<NSL>& sh, int lane, int& newton, double* A, double* Lp) {
  constexpr int RK = sym_rank<NS>();
  double* gs = &sh.g[0][lane];
  double* ws = &sh.w[0][lane];
  double det_Fp0;
  {
    double Fp0[9], invFp0[9], F[9];
    MpPtr q = fresh(m);
    m_load_start(q->Fp0, q->sub + SUB_FP0 * ln.sN, started, ln, Fp0);
    sub_F(m, Ftarget, started, ln, step, F);
    if (m_invert(Fp0, invFp0)) return ST_FAIL_STRESS;
    m_mul(F, invFp0, A);
    det_Fp0 = m_det(Fp0);
  }
  {
    double S0[9], s[6], x0[NSL];
    unsigned posm;
    MpPtr q = fresh(m);
    ld_start<NSL>(q->xi0, q->st0s, started, ln, 0, x0);
    m_load(s_cur ? q->S : q->S0, ln, S0);
#pragma unroll
    for (int r = 0; r < NSL; r++) ws[r * SWG] = dmk_rcp(x0[r]);
    sym_proj<RK>(S0, s);
    kinetics<NSL, QP, NS, false>(ph, s, ws, gs, nullptr, nullptr, posm);
    if (dot_state<NSL, QP>(ph, [&](int r) { return x0[r]; }, gs, ws)) return ST_FAIL_STATE;
    MpPtr q2 = fresh(m);
#pragma unroll
    for (int r = 0; r < NSL; r++) {
      const double dx = ws[r * SWG];
      st(q2->last1, ln, r, dx);
      st(q2->last1, ln, NSL + r, gs[r * SWG]);
      ws[r * SWG] = dmk_rcp(fma(dx, dt, x0[r]));
    }
  }
  bool cur = false;                   // last1 holds dotState_last(:,1) when !cur (uniform in the wavefront)
  for (int it = 1; it <= num.N_iter_state_max; it++) {
    sh.fpi[lane]++;
    const int status = integrate_stress<NSL, QP, NS>(ph, num, A, det_Fp0, dt, sh, lane, newton, Lp);
    if (status != ST_OK) return status;
    MpPtr q = fresh(m);
    const double* w1p = cur ? q->last2 : q->last1;
    double* w2p = cur ? q->last1 : q->last2;
    double w1[2 * NSL], w2[2 * NSL], s0[2 * NSL];
#pragma unroll
    for (int r = 0; r < NSL; r++) w1[r] = ld(w1p, ln, r);
    ld_start<NSL>(q->xi0, q->st0s, started, ln, 0, s0);
    // the converged Newton iterate evaluated kinetics_sl at this (S, xi): rates
    // are in gs.  A NaN rate ends the iteration with the status of the stress
    // integration, as the reference's exit does (phase_mechanical.f90:638)
    const bool nan = dot_state<NSL, QP>(ph, [&](int r) { return fma(w1[r], dt, s0[r]); }, gs, ws);
#pragma unroll
    for (int r = NSL; r < 2 * NSL; r++) w1[r] = ld(w1p, ln, r);
    ld_start<NSL>(q->gam0, q->st0s + NSL * ln.sN, started, ln, 0, s0 + NSL);
#pragma unroll
    for (int r = 0; r < 2 * NSL; r++) w2[r] = 0.0;
    if (it > 1) {
#pragma unroll
      for (int r = 0; r < 2 * NSL; r++) w2[r] = ld(w2p, ln, r);
    }
    // damper (src/phase_mechanical.f90:653-674)
    double d12 = 0.0, d22 = 0.0, d01 = 0.0;
#pragma unroll
    for (int r = 0; r < 2 * NSL; r++) {
      const double d0 = r < NSL ? ws[r * SWG] : gs[(r - NSL) * SWG], c = w1[r] - w2[r];
      d12 = fma(d0 - w1[r], c, d12);
      d22 = fma(c, c, d22);
      d01 = fma(d0, w1[r], d01);
    }
    const double zeta = (fmin(d01, d12) < 0.0 && d22 > 0.0) ? 0.75 + 0.25 * tanh_ool(2.0 + 4.0 * d12 / d22) : 1.0;
    MpPtr q3 = fresh(m);
    bool conv = true;
    // the next iterate start + dt d, d the damped rate: it differs from the last
    // one, start + dt w1, by the residual dt (w1 - d).  With a NaN rate the state
    // stays the last iterate.
#pragma unroll
    for (int r = 0; r < 2 * NSL; r++) {
      const double d0 = r < NSL ? ws[r * SWG] : gs[(r - NSL) * SWG];
      const double d = nan ? w1[r] : d0 * zeta + w1[r] * (1.0 - zeta);
      st(w2p, ln, r, d);               // dotState_last(:,1) of the next iteration
      const double s = fma(d, dt, s0[r]), res = (w1[r] - d) * dt;
      conv = conv && (fabs(res) <= fmax(r < NSL ? ph->atol_xi : ph->atol_gamma, num.eps_rel_state * fabs(s)));
      if (r < NSL) {
        st(q3->xi, ln, r, s);
        ws[r * SWG] = dmk_rcp(s);      // for the next stress integration
      } else {
        st(q3->gam, ln, r - NSL, s);
      }
    }
    cur = !cur;
    if (nan || conv) return ST_OK;
  }
  return ST_FAIL_STATE;
}

// one material point update per lane: block `blk` of the cells of m
template <int NSL, bool QP, bool NS>
DI void stress_body(MpPtr m, const double* __restrict__ Ftarget, PhPtr ph, int phase_id,
                    const DmkNumMech& num, double dt, int blk, SlipLds<NSL>& sh) {
  const int lane = threadIdx.x;
  const int e = blk * SWG + lane;
  if (e >= m->N) return;
  if (m->phase[e] != phase_id) return;
  const Lane ln = make_lane(m->N, e);

  // isostrain partition (src/homogenization_mechanical_isostrain.f90:60-75)
  {
    double F[9];
    m_load(Ftarget, ln, F);
    m_store(m->Fphase, ln, F);
  }
  // start values of the sub-step: those of the converged increment until a
  // sub-step completes (started), then copies in the sub-step scratch / st0s;
  // the initial state rate is taken at S_0 until a sub-step completes, then at
  // the last completed sub-step's S (s_cur)
  bool started = false, s_cur = false;
  // the last L_p (phase_mechanical_Lp is not restored between calls) and
  // A = F F_p0^-1 of the sub-step in progress
  double Lp[9], A[9];
  m_load(m->Lp, ln, Lp);
#pragma unroll
  for (int k = 0; k < 9; k++) A[k] = 0.0;

  int newton = 0;
  sh.fpi[lane] = 0;
  sh.nsub[lane] = 0;
  // phase_mechanical_constitutive substepping; the first pass takes the
  // cut-back branch, which is phase_restore (src/phase_mechanical.f90:1096-1115)
  sh.frac[lane] = 0.0;
  sh.step[lane] = 1.0 / num.r_cutback;
  int status = ST_ITERATING;
  bool todo = true;
  while (todo) {
    if (status == ST_OK) {
      const double done = sh.step[lane], stepFrac = sh.frac[lane] + done;
      const double step = fmin(1.0 - stepFrac, num.r_increase * done);
      sh.frac[lane] = stepFrac;
      todo = step > 0.0;
      if (todo) {
        // the completed sub-step's F, F_p, L_p and state are the next one's start
        double F[9];
        sub_F(m, Ftarget, started, ln, done, F);
        MpPtr q = fresh(m);
        double* sub = q->sub;
        finish_point<false>(ph, m, ln, started, A, Lp, done * dt, sub + SUB_FP0 * ln.sN);
        m_store(sub + SUB_F0 * ln.sN, ln, F);
        m_store(sub + SUB_LP0 * ln.sN, ln, Lp);
#pragma unroll 1
        for (int r = 0; r < NSL; r++) {
          st(q->st0s, ln, r, ld(q->xi, ln, r));
          st(q->st0s, ln, NSL + r, ld(q->gam, ln, r));
        }
        sh.step[lane] = step;
        started = true;
        s_cur = true;
      }
    } else {
      // cut back: restore the sub-step start (F_p, S = S_0, L_p for an actual
      // cut-back, state).  F_p, S and the state are outputs only until they are
      // read again, so they are restored where they are read: the state
      // integration starts from the sub-step start / S_0
      const double step = num.r_cutback * sh.step[lane];
      sh.step[lane] = step;
      s_cur = false;
      if (step < 1.0) {
        MpPtr q = fresh(m);
        m_load_start(q->Lp0, q->sub + SUB_LP0 * ln.sN, started, ln, Lp);
      }
      todo = step > num.r_cutback_min;
    }
    if (todo) {
      status = integrate_state_fpi<NSL, QP, NS>(ph, num, m, Ftarget, ln, started, s_cur, sh.step[lane],
                                                sh.step[lane] * dt, sh, lane, newton, A, Lp);
      sh.nsub[lane]++;
    }
  }
  MpPtr q = fresh(m);
  m_store(q->Lp, ln, Lp);
  if (status == ST_OK) {
    finish_point<true>(ph, m, ln, started, A, Lp, sh.step[lane] * dt, q->Fp);
  } else {
    // the restored sub-step start, as the last cut-back left it
    double T[9];
    m_load_start(q->Fp0, q->sub + SUB_FP0 * ln.sN, started, ln, T);
    m_store(q->Fp, ln, T);
    m_load(q->S0, ln, T);
    m_store(q->S, ln, T);
#pragma unroll 1
    for (int r = 0; r < NSL; r++) {
      double v[2];
      ld_start<1>(q->xi0, q->st0s, started, ln, r, v);
      ld_start<1>(q->gam0, q->st0s + NSL * ln.sN, started, ln, r, v + 1);
      st(q->xi, ln, r, v[0]);
      st(q->gam, ln, r, v[1]);
    }
  }
  MpPtr q4 = fresh(m);
  q4->status[e] = status;
  q4->n_newton[e] = newton;
  q4->n_fpi[e] = sh.fpi[lane];
  q4->n_sub[e] = sh.nsub[lane];
}

// the arguments of stress_kernel, read through its kernel-argument segment
struct StressArgs {
  DmkMPDev mp;
  const double* F;
  const DmkPhaseDev* ph;
  DmkNumMech num;
  double dt;
  int phase_id;
};

template <int NSL, bool QP, bool NS>
__global__ void __launch_bounds__(SWG) __attribute__((amdgpu_waves_per_eu(stress_waves(NSL))))
stress_kernel(StressArgs a) {
  __shared__ SlipLds<NSL> sh;
  MpPtr m = (MpPtr)__builtin_amdgcn_kernarg_segment_ptr();   // a.mp, the first argument's first member
  stress_body<NSL, QP, NS>(m, a.F, (PhPtr)a.ph, a.phase_id, a.num, a.dt, blockIdx.x, sh);
}

// The stress integration of several RVEs (and phases) in one launch: item i
// owns blocks [block0_i, block0_{i+1}) and runs them on its own material
// point, phase tables, load and time step, exactly as stress_kernel would.
template <int NSL, bool QP, bool NS>
__global__ void __launch_bounds__(SWG) __attribute__((amdgpu_waves_per_eu(stress_waves(NSL))))
stress_kernel_batch(const DmkStressItem* __restrict__ items, int n_items) {
  __shared__ SlipLds<NSL> sh;
  const int b = blockIdx.x;
  int lo = 0, hi = n_items - 1;                     // last item with block0 <= b (uniform)
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (items[mid].block0 <= b) lo = mid; else hi = mid - 1;
  }
  const DmkStressItem* it = items + lo;
  const DmkNumMech num = it->num;
  stress_body<NSL, QP, NS>((MpPtr)&it->mp, it->F, (PhPtr)it->ph,
                           it->phase_id, num, it->dt, b - it->block0, sh);
}

// The rotation R of F = R U (math_rotationalPart, src/math.f90:1004-1043) as the
// limit of R <- (R + R^-T)/2 from F (Higham, SIAM J. Sci. Stat. Comput. 7(4) 1986),
// which converges quadratically: a step below 1e-8 leaves an error below 1e-16.
// An elastic F takes three steps.
DI void rotational_part(const double* F, double* R) {
#pragma unroll
  for (int k = 0; k < 9; k++) R[k] = F[k];
#pragma unroll 1
  for (int it = 0; it < 64; it++) {
    double c[9];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const int i1 = (i + 1) % 3, i2 = (i + 2) % 3, j1 = (j + 1) % 3, j2 = (j + 2) % 3;
        c[3 * i + j] = R[3 * i1 + j1] * R[3 * i2 + j2] - R[3 * i1 + j2] * R[3 * i2 + j1];
      }
    const double g = 0.5 * dmk_rcp(R[0] * c[0] + R[1] * c[1] + R[2] * c[2]);
    double d2 = 0.0;
#pragma unroll
    for (int k = 0; k < 9; k++) {
      const double d = fma(g, c[k], -0.5 * R[k]);
      d2 = fma(d, d, d2);
      R[k] += d;
    }
    if (!(d2 > 1.0e-16)) break;
  }
}

// om2qu (src/rotations.f90:486-514), P = -1: the largest of 4 q_k^2 (by the
// reference's comparisons) gives its component, which divides the others; the
// four cases share one root
DI void om2qu(const double* om, double* qu) {
  const double tr = om[0] + om[4] + om[8];
  const bool c0 = tr > 0.0, c1 = om[0] > om[4] && om[0] > om[8], c2 = om[4] > om[8];
  const double t = c0 ? tr + 1.0
                      : (c1 ? 1.0 + om[0] - om[4] - om[8]
                            : (c2 ? 1.0 + om[4] - om[0] - om[8] : 1.0 + om[8] - om[0] - om[4]));
  const double h = 0.5 * dmk_rsq(t), big = t * h;
  const double m0 = (om[7] - om[5]) * h, m1 = (om[2] - om[6]) * h, m2 = (om[3] - om[1]) * h;
  const double p0 = (om[5] + om[7]) * h, p1 = (om[2] + om[6]) * h, p2 = (om[1] + om[3]) * h;
  qu[0] = c0 ? big : (c1 ? m0 : (c2 ? m1 : m2));
  qu[1] = c0 ? m0 : (c1 ? big : (c2 ? p2 : p1));
  qu[2] = c0 ? m1 : (c1 ? p2 : (c2 ? big : p0));
  qu[3] = c0 ? m2 : (c1 ? p1 : (c2 ? p0 : big));
  if (signbit(qu[0])) for (int k = 0; k < 4; k++) qu[k] = -qu[k];
  for (int k = 1; k < 4; k++) if (!dEq0(qu[k])) qu[k] = -qu[k];
  const double n = dmk_rsq(qu[0] * qu[0] + qu[1] * qu[1] + qu[2] * qu[2] + qu[3] * qu[3]);
  for (int k = 0; k < 4; k++) qu[k] *= n;
}

// row r (runtime, uniform) of a register 3x3 without dynamic register indexing
DI void row3(const double* M, int r, double* v) {
#pragma unroll
  for (int j = 0; j < 3; j++) v[j] = r == 0 ? M[j] : (r == 1 ? M[3 + j] : M[6 + j]);
}

// A E_k B^T for the symmetric basis tensor E_k (k a compile-time constant)
DI void basis_between(const double* A, int k, const double* B, double* T) {
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const double* a = A + 3 * i;
      const double* b = B + 3 * m;
      double v;
      switch (k) {
        case 0: v = R2 * (a[0] * b[0] - a[1] * b[1]); break;
        case 1: v = R6 * (a[0] * b[0] + a[1] * b[1] - 2.0 * (a[2] * b[2])); break;
        case 2: v = R2 * (a[1] * b[2] + a[2] * b[1]); break;
        case 3: v = R2 * (a[0] * b[2] + a[2] * b[0]); break;
        case 4: v = R2 * (a[0] * b[1] + a[1] * b[0]); break;
        default: v = R3 * (a[0] * b[0] + a[1] * b[1] + a[2] * b[2]); break;
      }
      T[3 * i + m] = v;
    }
}

// a, b, c, d summed over the wavefront: every lane of the k-th row of 16 lanes
// holds the sum of the k-th.  Two swaps of half-waves and rows fold four values
// into one register, four rotations within the rows finish them: 21 instructions
// for four sums instead of 18 for each.
DI void swap_halves(double& a, double& b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  a = __hiloint2double(hi[0], lo[0]);
  b = __hiloint2double(hi[1], lo[1]);
}
DI void swap_rows(double& a, double& b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  a = __hiloint2double(hi[0], lo[0]);
  b = __hiloint2double(hi[1], lo[1]);
}
template <int ROR>
DI double row_ror(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x120 + ROR, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x120 + ROR, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
DI double wave_rows(double a, double b, double c, double d) {
  swap_halves(a, c);
  double s = a + c;       // lower half: a, upper half: c
  swap_halves(b, d);
  double t = b + d;
  swap_rows(s, t);
  s += t;                 // rows: a, b, c, d
  s += row_ror<8>(s);
  s += row_ror<4>(s);
  s += row_ror<2>(s);
  s += row_ror<1>(s);
  return s;
}

// Orientation and consistent tangent of the homogenization (one constituent,
// v = 1) for a response in which every cell converged (flag[0] == ST_OK).
// Also writes the squared Frobenius norm of each cell's dPdF and, with part, per
// work-group its 81 sums and the extrema of the norms (dmk_stiffness_averages),
// to which every phase adds its cells; reading dPdF again for the sums took 38 us
// at 64^3.
//
// Column (k, l): dS = dS/dF_kl solves dS + dt sum_a dg_a C:sym(G2 P_a) (P_nS_a : dS)
// = C:sym(X), X = F_e(k,:) (x) F_p^-1(l,:), G2 = F_e^T A2.  As in the stress
// integration the sum acts through the E coordinates z of dS alone: N z = C E:X with
// N_kl = delta_kl + dt C_k E_k : (G2 W_l), one 5x5 (6x6) factorisation for the
// nine columns; then t = sum_a dg_a P_a (P_nS_a : dS) = sum_l z_l W_l,
// dS = sum_k z_k E_k with z_6 = C_6 E_6 : (X - dt G2 t), and with
// D = -dt F_p0^-1 t the derivative of F_p^-1
//   dP = e_k (x) (F_p^-1 S F_p^-T)(l,:) + F (D S F_p^-T + F_p^-1 (dS F_p^-T + S D^T))
//      = e_k (x) (F_p^-1 S F_p^-T)(l,:) + sum_l z_l T_l,
// T_l = F F_p^-1 E_l F_p^-T - dt (F F_p0^-1 W_l S F_p^-T + F F_p^-1 S W_l^T F_p0^-T):
// the six T_l are formed once, a column is then a 5x5 solve and 54 products.
// The traffic (57 values a cell in, 86 out: 60 us at 64^3 at copy rate) and the
// latency of a wavefront's chain bound it: one wavefront a SIMD, all inputs loaded
// at once.  64^3 cells of the cF tension 116 us, with stiffness_averages 128; a
// column at a time, with the averages from dPdF, took 155 + 58 us.  Two
// wavefronts a SIMD, with spills: 134 us without the sums, against 98 us.
template <int NSL, bool QP, bool NS>
__global__ void __launch_bounds__(SWG) __attribute__((amdgpu_waves_per_eu(1)))
tangent_kernel(DmkMPDev mp, const DmkPhaseDev* __restrict__ ph_, int phase_id, double dt,
               const int* __restrict__ flag, double* __restrict__ dPdF, double* __restrict__ nrm,
               double* __restrict__ part, double* __restrict__ pmax, double* __restrict__ pmin) {
  constexpr int RK = sym_rank<NS>();
  PhPtr ph = (PhPtr)ph_;
  // [row][lane]: 1/xi and the rate derivatives per system; then W_l in rows 8 l to
  // 8 l + 7, where T_l (but its last entry) takes its place
  __shared__ double sh[(2 * NSL > 8 * RK ? 2 * NSL : 8 * RK)][SWG];
  __shared__ double sums[81];
  const int lane = threadIdx.x;
  if (flag[0] != ST_OK) return;
  // lanes without a cell of this phase go along, for the sums over the wavefront
  const int e = min((int)(blockIdx.x * SWG) + lane, mp.N - 1);
  const bool act = (int)(blockIdx.x * SWG) + lane < mp.N && mp.phase[e] == phase_id;
  const bool first = phase_id == 0;
  if (!__any(act)) {
    if (part && first) {
      for (int c = lane; c < 81; c += SWG) part[81l * blockIdx.x + c] = 0.0;
      if (lane == 0) { pmax[blockIdx.x] = 0.0; pmin[blockIdx.x] = DBL_MAX; }
    }
    return;
  }
  const Lane ln = make_lane(mp.N, e);
  double N[RK * RK], rd[RK], v0[RK], tau[RK], g6[RK];
  double T6[9], T8[RK];       // T_6 (Schmid law) and the last entries of T_1..T_RK
  // every input at once: one trip to memory
  double xi[NSL], S[9], Fp[9], Fp0[9], F[9], Fe[9];
#pragma unroll
  for (int r = 0; r < NSL; r++) xi[r] = ld(mp.xi, ln, r);
  m_load(mp.S, ln, S);
  m_load(mp.Fp, ln, Fp);
  m_load(mp.Fp0, ln, Fp0);
  m_load(mp.Fphase, ln, F);
  m_load(mp.Fe, ln, Fe);
  batch_end();
  double invFp[9], Mid[9];
  {
    double A2[9], invFp0[9], B[9], M1[9], BS[9];
    {
      double H[5][RK], K[3][RK], s[6], l5[5], k3[3];
      unsigned posm;
#pragma unroll
      for (int r = 0; r < NSL; r++) sh[r][lane] = dmk_rcp(xi[r]);
      sym_proj<RK>(S, s);
      kinetics<NSL, QP, NS, true>(ph, s, &sh[0][lane], &sh[NSL][lane], l5, k3, posm);
      slip_moments<NSL, NS>(ph, &sh[NSL][lane], 1.0, posm, H, K);
      m_invert(Fp, invFp);
      m_invert(Fp0, invFp0);
      m_mul(F, invFp0, A2);
#pragma unroll
      for (int q = 0; q < 9; q++) { A2[q] *= dt; invFp0[q] *= -dt; }
      m_mul(F, invFp, B);
      m_mul_nt(S, invFp, M1);          // S F_p^-T
      m_mul(invFp, M1, Mid);           // F_p^-1 S F_p^-T
      m_mul(B, S, BS);
      double G2[9];
      m_mul_tn(Fe, A2, G2);            // dt F_e^T A2
      reduced_matrix<RK>(ph, G2, H, K, N);
#pragma unroll
      for (int l = 0; l < RK; l++) {
        // W_l to LDS; tr(G2 W_l)/sqrt3
        double h[5], q3[3], W[9], v = 0.0;
#pragma unroll
        for (int k = 0; k < 5; k++) { h[k] = H[k][l]; sh[8 * l + k][lane] = h[k]; }
#pragma unroll
        for (int m = 0; m < 3; m++) { q3[m] = K[m][l]; sh[8 * l + 5 + m][lane] = q3[m]; }
        if (RK == 5) {
          from_basis(h, q3, W);
#pragma unroll
          for (int q = 0; q < 9; q++) v = fma(G2[(q % 3) * 3 + q / 3], W[q], v);
        }
        g6[l] = v * R3;
      }
    }
#pragma unroll
    for (int l = 0; l < RK; l++) {
      double h[5], k3[3], W[9], V[9], U[9], T[9];
#pragma unroll
      for (int k = 0; k < 5; k++) h[k] = sh[8 * l + k][lane];
#pragma unroll
      for (int m = 0; m < 3; m++) k3[m] = sh[8 * l + 5 + m][lane];
      from_basis(h, k3, W);
      basis_between(B, l, invFp, T);
      m_mul(W, M1, V);
      m_mul(A2, V, U);
#pragma unroll
      for (int q = 0; q < 9; q++) T[q] -= U[q];
      m_mul_nt(BS, W, V);
      m_mul_nt(V, invFp0, U);
#pragma unroll
      for (int q = 0; q < 9; q++) T[q] += U[q];
#pragma unroll
      for (int q = 0; q < 8; q++) sh[8 * l + q][lane] = T[q];
      T8[l] = T[8];
    }
    if (RK == 5) basis_between(B, 5, invFp, T6);
  }
  const bool sing = dmk_qr_factor<RK>(N, rd, v0, tau);
  const double C6 = ph->C11 + 2.0 * ph->C12;
  double n2 = 0.0;
#pragma unroll 1
  for (int l = 0; l < 3; l++) {
    double pl[3], ml[3], z[3][6];
    row3(invFp, l, pl);
    row3(Mid, l, ml);
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const double* fk = Fe + 3 * k;
      double X[9];
#pragma unroll
      for (int n = 0; n < 3; n++)
#pragma unroll
        for (int m = 0; m < 3; m++) X[3 * n + m] = fk[n] * pl[m];
      sym_proj<RK>(X, z[k]);
#pragma unroll
      for (int q = 0; q < RK; q++) z[k][q] *= modulus<RK>(ph, q);
      // (as after a failed solve where N is singular: dS = C:sym(X))
      if (!sing) dmk_qr_apply_solve<RK>(N, rd, v0, tau, z[k]);
      if (RK == 5) {
        double v = (X[0] + X[4] + X[8]) * R3;
        if (!sing) {
#pragma unroll
          for (int q = 0; q < RK; q++) v = fma(-g6[q], z[k][q], v);
        }
        z[k][5] = C6 * v;
      }
    }
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int i = 0; i < 3; i++) {
        const int c = 3 * i + j;
        double v[3];
#pragma unroll
        for (int q = 0; q < 6; q++) {
          const double t = q >= RK ? T6[c] : (c == 8 ? T8[q < RK ? q : 0] : sh[8 * q + (c & 7)][lane]);
#pragma unroll
          for (int k = 0; k < 3; k++) v[k] = q ? fma(z[k][q], t, v[k]) : z[k][0] * t;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
          if (i == k) v[k] += ml[j];
          if (act) st(dPdF, ln, i + 3 * j + 9 * k + 27 * l, v[k]);
          n2 = fma(v[k], v[k], n2);
          if (!act) v[k] = 0.0;
        }
        if (part) {
          // row k of 16 lanes: the sum of v[k]
          const double sum = wave_rows(v[0], v[1], v[2], 0.0);
          const int k = lane >> 4;
          if ((lane & 15) == 0 && k < 3) sums[i + 3 * j + 9 * k + 27 * l] = sum;
        }
      }
  }
  if (part) {
    __syncthreads();       // sums: written by lanes 0, 16 and 32, read by all
    double mx = act && n2 > 0.0 ? n2 : 0.0, mn = act && n2 < DBL_MAX ? n2 : DBL_MAX;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      mx = fmax(mx, __shfl_xor(mx, o, 64));
      mn = fmin(mn, __shfl_xor(mn, o, 64));
    }
    for (int c = lane; c < 81; c += SWG) {
      double* d = part + 81l * blockIdx.x + c;
      *d = first ? sums[c] : *d + sums[c];
    }
    if (lane == 0) {
      pmax[blockIdx.x] = first ? mx : fmax(mx, pmax[blockIdx.x]);
      pmin[blockIdx.x] = first ? mn : fmin(mn, pmin[blockIdx.x]);
    }
  }
  double R[9], Rt[9], q[4];
  rotational_part(Fe, R);
  m_transpose(R, Rt);
  om2qu(Rt, q);
  if (!act) return;
  nrm[e] = n2;
#pragma unroll
  for (int k = 0; k < 4; k++) st(mp.O, ln, k, q[k]);
}

}  // namespace

// ---------------------------------------------------------------------------- launchers
namespace {

// f(slip systems, quarter powers, non-Schmid terms) with compile-time arguments
// for a variant = nsl (+ DMK_SYS_NONSCHMID); false when there is no such kernel
template <bool B>
struct Flag { static constexpr bool value = B; };
template <int N>
struct Count { static constexpr int value = N; };

template <class Fn>
bool for_variant(int variant, bool qp, Fn&& f) {
  auto pick = [&](auto n) {
    const bool ns = variant >= DMK_SYS_NONSCHMID;
    if (qp) ns ? f(n, Flag<true>{}, Flag<true>{}) : f(n, Flag<true>{}, Flag<false>{});
    else ns ? f(n, Flag<false>{}, Flag<true>{}) : f(n, Flag<false>{}, Flag<false>{});
  };
  switch (variant % DMK_SYS_NONSCHMID) {
    case 12: pick(Count<12>{}); return true;
    case 24: pick(Count<24>{}); return true;
    default: return false;
  }
}

}  // namespace

extern "C" int dmk_launch_stress(const DmkMPDev* mp, const double* Ftarget, const DmkPhaseDev* ph,
                                 const DmkPhaseDev* ph_host, int phase_id, const DmkNumMech* num, double dt,
                                 hipStream_t s) {
  const dim3 blk(SWG), grd((mp->N + SWG - 1) / SWG);
  const bool known = for_variant(dmk_sys_variant(ph_host), ph_host->quarter_pow != 0, [&](auto n, auto qp, auto ns) {
    hipLaunchKernelGGL((stress_kernel<decltype(n)::value, decltype(qp)::value, decltype(ns)::value>), grd, blk, 0, s,
                       StressArgs{*mp, Ftarget, ph, *num, dt, phase_id});
  });
  if (!known) return 1;
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

extern "C" int dmk_launch_stress_batch(const DmkStressItem* items_dev, int n_items, int n_blocks, int variant,
                                       int quarter_pow, hipStream_t s) {
  if (n_items < 1 || n_blocks < 1) return 0;
  const dim3 blk(SWG), grd(n_blocks);
  const bool known = for_variant(variant, quarter_pow != 0, [&](auto n, auto qp, auto ns) {
    hipLaunchKernelGGL((stress_kernel_batch<decltype(n)::value, decltype(qp)::value, decltype(ns)::value>), grd, blk,
                       0, s, items_dev, n_items);
  });
  if (!known) return 1;
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

extern "C" int dmk_launch_tangent(const DmkMPDev* mp, const DmkPhaseDev* ph, const DmkPhaseDev* ph_host,
                                  int phase_id, double dt, const int* flag, double* dPdF, double* nrm,
                                  double* part, double* pmax, double* pmin, hipStream_t s) {
  const dim3 blk(SWG), grd((mp->N + SWG - 1) / SWG);
  const bool known = for_variant(dmk_sys_variant(ph_host), ph_host->quarter_pow != 0, [&](auto n, auto qp, auto ns) {
    hipLaunchKernelGGL((tangent_kernel<decltype(n)::value, decltype(qp)::value, decltype(ns)::value>), grd, blk, 0, s,
                       *mp, ph, phase_id, dt, flag, dPdF, nrm, part, pmax, pmin);
  });
  if (!known) return 1;
  return hipGetLastError() == hipSuccess ? 0 : 2;
}

extern "C" int dmk_pow_law(const double* x, const double* y, double* out, int32_t n, int32_t quarter) {
  if (!x || !y || !out || n < 1) { dmk_set_error("dmk_pow_law: invalid argument"); return DMK_ERR_ARG; }
  if (quarter)
    for (int i = 0; i < n; i++)
      if (!(y[i] > 0.0 && y[i] <= 64.0 && y[i] * 4.0 == std::rint(y[i] * 4.0))) {
        dmk_set_error("dmk_pow_law: quarter-power exponents are positive multiples of 1/4 up to 64");
        return DMK_ERR_ARG;
      }
  double* d = nullptr;
  const size_t b = sizeof(double) * (size_t)n;
  if (hipMalloc((void**)&d, 3 * b) != hipSuccess) { hipGetLastError(); dmk_set_error("dmk_pow_law: device memory"); return DMK_ERR_HIP; }
  int rc = 0;
  if (hipMemcpy(d, x, b, hipMemcpyHostToDevice) != hipSuccess || hipMemcpy(d + n, y, b, hipMemcpyHostToDevice) != hipSuccess)
    rc = DMK_ERR_HIP;
  if (!rc) {
    const unsigned nb = (unsigned)((n + 255) / 256);
    if (quarter) hipLaunchKernelGGL(pow_law_kernel<true>, dim3(nb), dim3(256), 0, 0, d, d + n, d + 2 * n, n);
    else hipLaunchKernelGGL(pow_law_kernel<false>, dim3(nb), dim3(256), 0, 0, d, d + n, d + 2 * n, n);
    if (hipGetLastError() != hipSuccess || hipMemcpy(out, d + 2 * n, b, hipMemcpyDeviceToHost) != hipSuccess)
      rc = DMK_ERR_HIP;
  }
  hipFree(d);
  if (rc) dmk_set_error("dmk_pow_law: launch or copy failed");
  return rc;
}

enum { DMK_POWER_RATES = 0, DMK_POWER_HARDENING = 1, DMK_POWER_LIBRARY = 2 };   // path of dmk_power_laws

// CH values of x a thread, as the per-cell kernels power CH systems at once
__global__ void power_laws_kernel(const double* __restrict__ x, double y, int path, double* __restrict__ out, int n) {
  const int i0 = (blockIdx.x * blockDim.x + threadIdx.x) * CH, k = (int)(4.0 * y);
  if (i0 >= n) return;
  double v[CH], r[CH];
#pragma unroll
  for (int j = 0; j < CH; j++) {
    v[j] = i0 + j < n ? x[i0 + j] : 1.0;
    r[j] = path == DMK_POWER_LIBRARY ? v[j] : fabs(v[j]);
  }
  if (path == DMK_POWER_RATES) {
    quarter_power<CH>(r, k - 4);
#pragma unroll
    for (int j = 0; j < CH; j++) r[j] *= v[j];
  } else if (path == DMK_POWER_HARDENING) {
    quarter_power<CH>(r, k);
  } else {
#pragma unroll
    for (int j = 0; j < CH; j += 4) {
      Four a, e;
#pragma unroll
      for (int q = 0; q < 4; q++) { a.v[q] = r[j + q]; e.v[q] = y; }
      a = pow4_ool(a, e);
#pragma unroll
      for (int q = 0; q < 4; q++) r[j + q] = a.v[q];
    }
  }
#pragma unroll
  for (int j = 0; j < CH; j++)
    if (i0 + j < n) out[i0 + j] = r[j];
}

extern "C" int dmk_power_laws(const double* x, double* out, int32_t n, double y, int32_t path) {
  const bool quarter = path == DMK_POWER_RATES || path == DMK_POWER_HARDENING;
  if (!x || !out || n < 1 || (!quarter && path != DMK_POWER_LIBRARY) ||
      (quarter && !(y > 0.0 && y <= 64.0 && y * 4.0 == std::rint(y * 4.0))) || (path == DMK_POWER_RATES && y < 1.0)) {
    dmk_set_error("dmk_power_laws: invalid argument");
    return DMK_ERR_ARG;
  }
  const size_t b = sizeof(double) * (size_t)n;
  double* d = nullptr;
  if (hipMalloc((void**)&d, 2 * b) != hipSuccess) { hipGetLastError(); dmk_set_error("dmk_power_laws: device memory"); return DMK_ERR_HIP; }
  int rc = hipMemcpy(d, x, b, hipMemcpyHostToDevice) == hipSuccess ? 0 : DMK_ERR_HIP;
  if (!rc) {
    const unsigned nb = (unsigned)((n + 64 * CH - 1) / (64 * CH));
    hipLaunchKernelGGL(power_laws_kernel, dim3(nb), dim3(64), 0, 0, d, y, path, d + n, n);
    if (hipGetLastError() != hipSuccess || hipMemcpy(out, d + n, b, hipMemcpyDeviceToHost) != hipSuccess) rc = DMK_ERR_HIP;
  }
  hipFree(d);
  if (rc) dmk_set_error("dmk_power_laws: launch or copy failed");
  return rc;
}
