"""Algorithmic FLOP counts of the per-cell kernels, derived from the operations
the stress-integration kernel performs (a fused multiply-add counts 2, a
division, square root or pow counts 1).  The counts multiply device-side
iteration counters (Newton iterations, state-integrator iterations) to give
the FLOPs of one response.

Newton iteration of integrateStress (N_sl slip systems, Schmid law), per cell:
  F_e = A - dt (A L_p)                           63
  S: F_e^T F_e - I, coordinates                  43
  kinetics: tau (5 products) 9, ratio, pow, rate and derivative 6, L_p (8 FMA) 16     32 N_sl
  L_p from coordinates, residual, norms          79
  sum u q x P: 15 symmetric + 15 skew FMA, factors                                    66 N_sl
  G = F_e^T A                                    45
  reduced 5x5 matrix (5 products G W_l)          370
  right-hand side                                55
  5x5 Householder QR and solve                   270
  x = res - sum y_l W_l, step                    107
State-integrator iteration (beyond its Newton iterations):
  rates from derivatives 11, 1 - xi / xi_sat, pow, h 6, hardening row 2 N_sl + 1, damper and update
  (18 per state entry, 2 N_sl entries) 36, 1/xi 1, per system; determinants, zeta 45; half of the
  prologue and epilogue (F_p0^-1, A, F_p, S, P: 400 a cell, about two iterations) 200
Tangent kernel (once per cell and response): kinetics 32 N_sl, moments 66 N_sl; inverses and
  products of 3x3 360; reduced matrix 370, traces 175, QR 167; T_l 1350; 9 columns of (right-hand
  side 20, solve 100, z_6 20, 6-term sums 108, norm 18); rotation 250.
"""


def newton_flops(nsl: int) -> int:
    return 63 + 43 + 79 + 45 + 370 + 55 + 270 + 107 + 98 * nsl


def state_flops(nsl: int) -> int:
    return nsl * (2 * nsl + 55) + 245


def tangent_flops(nsl: int) -> int:
    return 98 * nsl + 360 + 370 + 175 + 167 + 1350 + 9 * 266 + 250


def stress_kernel_flops(nsl: int, newton_iterations: int, state_iterations: int) -> int:
    return newton_flops(nsl) * newton_iterations + state_flops(nsl) * state_iterations


# Algorithmic HBM bytes per cell of the stress kernel: read F, F0, F_p0, L_p0,
# S0 (5 x 72), xi0, gamma0 (2 N_sl x 8); write F_phase, P, S, L_p, F_p, F_e
# (6 x 72), xi, gamma (2 N_sl x 8), status/counters (12)
def stress_kernel_bytes(nsl: int) -> int:
    return 5 * 72 + 16 * nsl + 6 * 72 + 16 * nsl + 12


# Per residual evaluation of the spectral part (N cells, Nk = (N1/2+1) N2 N3):
def spectral_bytes(N: int, Nk: int) -> dict:
    return {"fft_fwd": 9 * N * 8 + 9 * Nk * 16, "gamma_div": 2 * 9 * Nk * 16, "fft_inv": 9 * Nk * 16 + 9 * N * 8}
