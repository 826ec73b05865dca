"""The gradient's sensitivity to rounding: a last-bit change of the cotangent
changes it by rounding only.  The reverse sweep's own rounding is 2e-14 of each
component on this case (measured over linear-solver tolerances 1e-8 to 1e-15);
1e-11 leaves room for another order of its sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_gradient_of_perturbed_cotangent(gpu_lib):
    from damask_amd import adjoint, config, workloads
    grid, mat = workloads.polycrystal([8, 8, 8], 4, 3)
    mat = config.parse_material(mat)
    _, lcs = config.parse_load(workloads.tension_x(8.0, 3))
    s, P = adjoint.run_curve(grid, mat, lcs)
    Pb = np.zeros_like(P)
    Pb[:, 0, 0] = -0.01 * P[:, 0, 0]
    g, _ = adjoint.curve_gradient(s, 0, Pb)
    bit = 1.0 + np.array([2.3e-16, -2.3e-16, 4.5e-16])[:, None, None]
    h, _ = adjoint.curve_gradient(s, 0, Pb * bit)
    s.close()
    assert (np.abs(h - g) <= 1e-11 * np.abs(g)).all(), np.abs(h / g - 1.0).max()
