"""Dot products of a residual evaluation where jobs share a block or not.

Sizes: less than a chunk of 2048 values; chunks enough for one, a few and all
jobs of a block (the rule takes chunks x jobs / 1024 jobs a block).  The dot
products steer the iteration only, so the converged P of a run equals that of a
run without acceleration (Richardson) within what both leave of the divergence,
1e-5 of the stress at wavelengths of a few cells, over 2 pi times the cells' size
in wavelengths: below 1e-4 of the largest stress."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [[5, 4, 3], [32, 32, 16], [48, 48, 50]])
def test_accelerated_equals_plain_iteration(gpu_lib, cells):
    from damask_amd import config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal(cells, 6, 2)
    mat = config.parse_material(mat)
    lc = config.parse_load(workloads.tension_x(1.0, 2))[1][0]
    P = []
    for solver in (0, 1):
        num = config.Numerics(solver=solver, eps_rel_div=1e-5)
        g = GridMechSpectralBasic(grid, mat, num)
        assert g.run_loadcase(lc)["rc"] == 0
        P.append(g.field("P"))
    assert np.abs(P[0] - P[1]).max() <= 1e-4 * np.abs(P[1]).max()
