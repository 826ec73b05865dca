"""Kernel variants of the material-point response against the oracle: exponents
shared by all systems or not, multiples of 1/4 or not, n below 1, work-groups of
one cell, a whole wavefront and a remainder, 12 and 24 systems, with and without
non-Schmid terms.

The stress iterations of both sides stop at 1e-6 of L_p and the state iterations
at 1e-6 of the state, so points agree within 1e-6 and, Newton's last step being
quadratic, averages within 1e-8."""
import copy

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _phase(lattice, n, a, non_schmid):
    from damask_amd import workloads
    p = copy.deepcopy(workloads.FCC_PHASE if lattice == "cF" else
                      (workloads.BCC_NS_STRONG_PHASE if non_schmid else workloads.BCC_PHASE))
    pl = p["mechanical"]["plastic"]
    pl["n_sl"], pl["a_sl"] = list(n), list(a)
    if lattice == "cI" and len(n) == 1:      # the {110}<111> family alone: 12 systems
        for k in ("N_sl", "dot_gamma_0_sl", "h_0_sl-sl", "xi_0_sl", "xi_inf_sl"):
            pl[k] = pl[k][:1]
    return p


@pytest.mark.parametrize("cells", [[1, 1, 1], [4, 4, 4], [13, 5, 1]])
@pytest.mark.parametrize("lattice,n,a,non_schmid", [
    ("cF", [20.0], [2.25], False),           # one powering for all systems
    ("cF", [20.25], [2.0], False),           # x^(1/4) base
    ("cF", [10.5], [1.0], False),            # x^(1/2) base
    ("cF", [1.0], [0.75], False),            # x^0: linear viscous
    ("cF", [0.75], [2.5], False),            # quarter powers, n < 1: one system at a time
    ("cF", [17.3], [2.1], False),            # library pow
    ("cI", [20.0, 20.0], [2.0, 2.0], False),
    ("cI", [20.0, 12.0], [2.0, 1.5], False),  # families with exponents of their own
    ("cI", [15.5, 11.1], [2.0, 2.0], False),
    ("cI", [20.0], [2.0], True),             # 12 systems, non-Schmid terms
    ("cI", [20.0, 20.0], [2.0, 2.0], True),
    ("cI", [20.0, 16.0], [2.0, 1.25], True),
    ("cI", [20.0], [2.1], True),             # library pow; n integer: a resolved stress may be negative in both senses
    ("cI", [20.0, 20.0], [2.0, 2.1], True),
])
def test_response_variants(gpu_lib, oracle, lattice, n, a, non_schmid, cells):
    from damask_amd import config, workloads
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal(cells, 3, 5, phase=_phase(lattice, n, a, non_schmid))
    mat = config.parse_material(mat)
    g = GridMechSpectralBasic(grid, mat, Numerics())
    o = oracle.Problem(grid, mat, Numerics())
    L, N, dt = oracle.lib(), grid.n_cells, 0.5
    rng = np.random.default_rng(3)
    eps = 2.5e-3 if non_schmid else 8e-4
    for step in range(1, 4):
        F = np.eye(3) + step * np.diag([eps, -0.4 * eps, -0.4 * eps]) + 0.1 * eps * rng.standard_normal((N, 3, 3))
        P_g, Pav_g, _, _, st_g = g.constitutive(F, dt)
        Ff = np.ascontiguousarray(F.transpose(0, 2, 1).reshape(-1))
        P_o, dP_o = np.zeros_like(Ff), np.zeros(81 * N)
        st_o = L.orc_mp_response(o.mp, dt, oracle.ptr(Ff), oracle.ptr(P_o), oracle.ptr(dP_o))
        assert st_g == st_o == 0
        P_o = P_o.reshape(-1, 3, 3).transpose(0, 2, 1)
        assert (np.abs(P_g - P_o).max(axis=(1, 2)) / np.abs(P_o).max(axis=(1, 2))).max() < 1e-6
        assert np.abs(Pav_g - P_o.mean(0)).max() < 1e-8 * np.abs(P_o.mean(0)).max()
        assert np.abs(g.field("dPdF") - dP_o.reshape(N, 81)).max() < 1e-6 * np.abs(dP_o).max()
        for name, what in (("xi_sl", 8), ("gamma_sl", 9)):
            x = g.field(name)
            y = o.get(what, x.shape[1]).reshape(N, -1)
            assert np.abs(x - y).max() <= 1e-8 * np.abs(y).max(), name
        g.materialpoint_forward()
        L.orc_mp_forward(o.mp)
    g.close()
