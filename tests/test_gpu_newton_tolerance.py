"""A tolerance of the stress iteration whose square underflows (norms are compared
squared): an unloaded point converges at once.  Its stress is the rounding of F_e, a few
1e-16 times a stiffness of 2e11 Pa, and the slip rates of that, (1e-12)^20, have squares of 0."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eps", [1.0e-8, 1.0e-200])
def test_unloaded_point(gpu_lib, eps):
    from damask_amd import config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal([4, 4, 4], 3, 5)
    g = GridMechSpectralBasic(grid, config.parse_material(mat), config.Numerics(eps_abs_Lp=eps))
    P, _, _, _, status = g.constitutive(np.tile(np.eye(3), (grid.n_cells, 1, 1)), 0.5)
    assert status == 0 and np.abs(P).max() < 1e-3
    g.close()
