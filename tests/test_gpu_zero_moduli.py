"""Phases with a zero elastic modulus (no shear stiffness, C_11 = C_12, no stiffness
at all) respond as the oracle's do.  Points agree within the 1e-6 at which both
sides' stress and state iterations stop."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("non_schmid", [False, True])
@pytest.mark.parametrize("moduli", [{"C_44": 0.0}, {"C_12": 1.0e11, "C_11": 1.0e11}, {"C_11": 0.0, "C_12": 0.0, "C_44": 0.0}])
def test_response(gpu_lib, oracle, moduli, non_schmid):
    from damask_amd import config, workloads
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    base = workloads.BCC_NS_STRONG_PHASE if non_schmid else workloads.FCC_PHASE
    soft = copy.deepcopy(base)
    soft["mechanical"]["elastic"].update(moduli)
    # every second grain soft: the average stiffness, which the solver sets up with, stays regular
    grid, mat = workloads.polycrystal([5, 4, 4], 4, 5, phase=base)
    name = mat["material"][0]["constituents"][0]["phase"]
    mat["phase"] = {name: base, "soft": soft}
    for m in mat["material"][::2]:
        m["constituents"][0]["phase"] = "soft"
    mat = config.parse_material(mat)
    g, o, L = GridMechSpectralBasic(grid, mat, Numerics()), oracle.Problem(grid, mat, Numerics()), oracle.lib()
    N = grid.n_cells
    rng = np.random.default_rng(3)
    eps = 2.5e-3 if non_schmid else 8e-4
    for step in range(1, 4):
        F = np.eye(3) + step * np.diag([eps, -0.4 * eps, -0.4 * eps]) + 0.1 * eps * rng.standard_normal((N, 3, 3))
        P, Pav, _, _, status = g.constitutive(F, 0.5)
        Ff = np.ascontiguousarray(F.transpose(0, 2, 1).reshape(-1))
        P_o, dP_o = np.zeros_like(Ff), np.zeros(81 * N)
        assert L.orc_mp_response(o.mp, 0.5, oracle.ptr(Ff), oracle.ptr(P_o), oracle.ptr(dP_o)) == 0
        assert status == 0
        P_o = P_o.reshape(-1, 3, 3).transpose(0, 2, 1)
        assert (np.abs(P - P_o).max(axis=(1, 2)) <= 1e-6 * np.abs(P_o).max(axis=(1, 2))).all()
        assert np.abs(g.field("dPdF") - dP_o.reshape(N, 81)).max() < 1e-6 * np.abs(dP_o).max()
        g.materialpoint_forward()
        L.orc_mp_forward(o.mp)
    g.close()
