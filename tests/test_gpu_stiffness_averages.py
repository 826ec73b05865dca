"""C_volAvg and C_minMaxAvg of the tangent pass against the same averages of its
dPdF field: work-groups of one cell, a whole wavefront and a remainder, one phase
and two phases sharing work-groups.

C_volAvg sums N positive and negative entries in another order: within N eps of
the mean absolute value.  C_minMaxAvg is half the sum of two cells' dPdF, the same
arithmetic on the same numbers, once the cells are the same; their norms differ
here by far more than rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [[1, 1, 1], [4, 4, 4], [13, 5, 1], [16, 16, 17]])
@pytest.mark.parametrize("dual", [False, True])
def test_averages_of_the_field(gpu_lib, cells, dual):
    from damask_amd import config, workloads
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal(cells, 5, 3)
    if dual:
        mat["phase"] = {**mat["phase"], "bcc": workloads.BCC_PHASE}
        for m in mat["material"][::2]:
            m["constituents"][0]["phase"] = "bcc"
    g = GridMechSpectralBasic(grid, config.parse_material(mat), Numerics())
    rng = np.random.default_rng(1)
    F = np.eye(3) + 4e-4 * np.diag([1.0, -0.4, -0.4]) + 2e-4 * rng.standard_normal((grid.n_cells, 3, 3))
    _, _, avg, cmm, status = g.constitutive(F, 0.5)
    assert status == 0
    dP = g.field("dPdF").reshape(grid.n_cells, 81)
    avg, cmm = avg.reshape(-1, order="F"), cmm.reshape(-1, order="F")
    tol = 4.0 * np.finfo(float).eps * (64 + grid.n_cells) * np.abs(dP).mean(axis=0)
    assert (np.abs(avg - dP.mean(axis=0)) <= tol).all()
    n2 = (dP * dP).sum(axis=1)
    assert (cmm == 0.5 * (dP[n2.argmax()] + dP[n2.argmin()])).all()
