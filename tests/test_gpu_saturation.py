"""Hardening at the ends of 1 - xi / xi_sat: without saturation (an infinite
xi_inf) the response is the oracle's; without hardening (xi_0 = xi_inf) it is exactly
zero, so that xi stays what it was for any exponent a_sl.  The exponents below 1 make
a rounding of 2e-16 in it a visible rate, and 1 / (xi (1 / xi)) is not 1 for the stresses chosen.

Points agree with the oracle within the 1e-6 at which both sides' stress and state iterations
stop."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(cells, lattice, **plastic):
    from damask_amd import config, workloads
    p = copy.deepcopy(workloads.FCC_PHASE if lattice == "cF" else workloads.BCC_PHASE)
    pl = p["mechanical"]["plastic"]
    for k, v in plastic.items():
        pl[k] = [v] * len(pl["n_sl"])
    grid, mat = workloads.polycrystal(cells, 3, 5, phase=p)
    return grid, config.parse_material(mat)


def _fields(N, steps=3):
    rng = np.random.default_rng(3)
    eps = 8e-4
    for step in range(1, steps + 1):
        yield np.eye(3) + step * np.diag([eps, -0.4 * eps, -0.4 * eps]) + 0.1 * eps * rng.standard_normal((N, 3, 3))


@pytest.mark.parametrize("lattice", ["cF", "cI"])
@pytest.mark.parametrize("a", [2.25, 0.75, 1.3])
def test_no_saturation(gpu_lib, oracle, lattice, a):
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = _problem([5, 4, 4], lattice, a_sl=a, xi_inf_sl=float("inf"))
    g, o, L = GridMechSpectralBasic(grid, mat, Numerics()), oracle.Problem(grid, mat, Numerics()), oracle.lib()
    N = grid.n_cells
    xi = [g.field("xi_sl")]
    for F in _fields(N):
        P, _, _, _, status = g.constitutive(F, 0.5)
        Ff = np.ascontiguousarray(F.transpose(0, 2, 1).reshape(-1))
        P_o, dP_o = np.zeros_like(Ff), np.zeros(81 * N)
        assert L.orc_mp_response(o.mp, 0.5, oracle.ptr(Ff), oracle.ptr(P_o), oracle.ptr(dP_o)) == 0
        assert status == 0
        P_o = P_o.reshape(-1, 3, 3).transpose(0, 2, 1)
        assert (np.abs(P - P_o).max(axis=(1, 2)) / np.abs(P_o).max(axis=(1, 2))).max() < 1e-6
        xi.append(g.field("xi_sl"))
        y = o.get(8, xi[-1].shape[1]).reshape(N, -1)
        assert np.abs(xi[-1] - y).max() <= 1e-8 * np.abs(y).max()
        g.materialpoint_forward()
        L.orc_mp_forward(o.mp)
    assert (xi[-1] > xi[0]).any()
    g.close()


@pytest.mark.parametrize("lattice", ["cF", "cI"])
@pytest.mark.parametrize("a", [0.25, 0.3])
@pytest.mark.parametrize("xi", [28.0e6, 56.0e6, 67.0e6, 83.0e6])
def test_no_hardening(gpu_lib, lattice, a, xi):
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = _problem([5, 4, 4], lattice, a_sl=a, xi_0_sl=xi, xi_inf_sl=xi)
    g = GridMechSpectralBasic(grid, mat, Numerics())
    for F in _fields(grid.n_cells):
        assert g.constitutive(F, 0.5)[4] == 0
        assert (g.field("xi_sl") == xi).all()
        g.materialpoint_forward()
    assert g.field("gamma_sl").max() > 1e-6
    g.close()
