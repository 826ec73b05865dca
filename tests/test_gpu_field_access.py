"""Fields to and from the host through the staging buffer: one and two cells, a
remainder of a tile, fields of nine values and wider ones, the stiffness through a
buffer of its own.  Values are moved, not computed, so they come back bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [[1, 1, 1], [2, 1, 1], [13, 5, 1], [17, 16, 5]])
@pytest.mark.parametrize("lattice", ["fcc", "bcc"])
def test_fields_round_trip(gpu_lib, cells, lattice):
    from damask_amd import config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    phase = workloads.FCC_PHASE if lattice == "fcc" else workloads.BCC_PHASE
    grid, mat = workloads.polycrystal(cells, 2, 1, phase=phase)
    g = GridMechSpectralBasic(grid, config.parse_material(mat), config.Numerics())
    rng = np.random.default_rng(0)
    for name in ("F", "F_p", "L_p", "S", "xi_sl", "gamma_sl"):
        v = rng.standard_normal(g.field(name).shape)
        g.set_field(name, v)
        assert (g.field(name) == v).all(), name
    F = np.broadcast_to(np.eye(3), (grid.n_cells, 3, 3))
    g2 = GridMechSpectralBasic(grid, config.parse_material(mat), config.Numerics())
    P, _, avg, _, status = g2.constitutive(F * (1.0 + 1e-5), 0.5)
    assert status == 0 and (g2.field("P") == P).all()
    assert np.allclose(g2.field("dPdF").mean(axis=0), avg.reshape(-1, order="F"), rtol=0,
                       atol=1e-12 * np.abs(avg).max())
