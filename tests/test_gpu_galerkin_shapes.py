"""The Galerkin scheme's convolution, even, odd and prime sizes, fused with the z
passes in one or two buffers and in passes of its own, against its formula in numpy: FP64 transforms of
few values, each output off by a few roundings per stage of the largest, well inside
1e-12 of it.  And the scheme, on whichever path its set-up picks, against the basic scheme:
both solve the same equilibrium, to 1e-6 of the stress in the divergence, which
leaves less than 1e-4 of the largest stress in a cell (1e-6 over 2 pi times a
wavelength of a few cells, times the contrast of the grains)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [[6, 5, 1], [5, 6, 7], [8, 8, 8], [6, 4, 13], [4, 6, 64]])
def test_galerkin_equals_basic(gpu_lib, cells):
    from damask_amd import config, workloads
    from damask_amd.grid import grid_mechanical
    grid, mat = workloads.polycrystal(cells, 3, 4)
    mat = config.parse_material(mat)
    lc = config.parse_load(workloads.tension_x(1.0, 2))[1][0]
    P = []
    for scheme in ("spectral_basic", "spectral_Galerkin"):
        g = grid_mechanical(scheme)(grid, mat, config.Numerics(eps_rel_div=1e-6, eps_rel_P=1e-6, eps_abs_P=1.0))
        assert g.run_loadcase(lc)["rc"] == 0
        P.append(g.field("P"))
    assert np.abs(P[0] - P[1]).max() <= 1e-4 * np.abs(P[0]).max()


@pytest.mark.parametrize("zgz", ["0", "1", "2"])
@pytest.mark.parametrize("cells", [[6, 5, 1], [5, 6, 7], [8, 8, 8], [6, 4, 13], [4, 6, 64], [3, 4, 192], [1, 6, 8]])
def test_convolution_against_numpy(gpu_lib, cells, zgz, monkeypatch):
    from damask_amd import _lib, config, workloads
    from damask_amd.grid import grid_mechanical
    monkeypatch.setenv("DMK_FFT_ZGZ", zgz)
    grid, mat = workloads.polycrystal(cells, 3, 4, size=(1.0, 0.9, 0.8))
    g = grid_mechanical("spectral_Galerkin")(grid, config.parse_material(mat), config.Numerics())
    path = g.scalar("fft_path")
    assert (path[2] > 0) == (zgz != "0" and cells[2] > 1)
    if path[2] > 0:
        assert path[4] == (zgz == "2" and cells[2] in (8, 64))
    x, y, z = cells
    f = np.random.default_rng(2).random((z, y, x, 3, 3))         # [..., m, l] = F_lm
    out = np.zeros(f.size)
    _lib.check(g.lib.dmk_galerkin_convolution(g.h, _lib.dptr(f.reshape(-1)), _lib.dptr(out)))
    Fh = np.fft.rfftn(f, axes=(0, 1, 2))
    a = np.zeros((z, y, x // 2 + 1, 3))
    for d, (n, axis) in enumerate(((x, 2), (y, 1), (z, 0))):
        k = np.arange(n // 2 + 1) if d == 0 else np.arange(n)
        k = np.where(k > n // 2, k - n, k).astype(float)
        if n % 2 == 0:
            k[n // 2] = 0.0
        a[..., d] = (2.0 * np.pi * k / grid.size[d]).reshape([-1 if i == axis else 1 for i in range(3)])
    n2 = (a * a).sum(-1)
    Fa = np.einsum("zyxol,zyxo->zyxl", Fh, a)                    # F_hat a
    G = -np.einsum("zyxm,zyxl->zyxml", a, Fa) / np.where(n2 > 1e-16, n2, 1.0)[..., None, None]
    G[n2 <= 1e-16] = 0.0
    G[0, 0, 0] = Fh[0, 0, 0]
    ref = np.fft.irfftn(G, s=(z, y, x), axes=(0, 1, 2)) * grid.n_cells
    assert np.abs(out.reshape(ref.shape) - ref).max() < 1e-12 * np.abs(ref).max()
    g.close()
