"""Transform shapes at the edges of the kernels' layouts: lines that 64 divides
(padded in LDS) next to lines it does not, the largest plane of the
single-buffer x-y kernels, odd radices and primes, lines of one.

FP64 transforms of at most 1e5 values against numpy's: each output is off by a few
roundings per stage of the largest, well inside 1e-12 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CELLS = [[128, 128, 2], [128, 64, 1], [64, 130, 1], [192, 6, 2], [320, 4, 1], [11, 13, 2], [22, 9, 3], [1, 64, 2],
         [2, 2, 64]]


def _solver(cells):
    from damask_amd import config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal(cells, 2, 1)
    return GridMechSpectralBasic(grid, config.parse_material(mat)), grid.n_cells


@pytest.mark.parametrize("xy", ["0", "1", "2"])
@pytest.mark.parametrize("cells", CELLS)
def test_transforms_against_numpy(gpu_lib, cells, xy, monkeypatch):
    from damask_amd import _lib
    monkeypatch.setenv("DMK_FFT_XY", xy)
    g, N = _solver(cells)
    if xy == "2" and cells[:2] == [128, 128]:
        assert g.scalar("fft_path")[1] == 1
    x, y, z = cells
    f = np.random.default_rng(2).random((z, y, x, 9))
    out = np.zeros(2 * 9 * (x // 2 + 1) * y * z)
    _lib.check(g.lib.dmk_fft_forward(g.h, 9, _lib.dptr(f.reshape(-1)), _lib.dptr(out)))
    ref = np.fft.rfftn(f, axes=(0, 1, 2))
    got = out.reshape(z, y, x // 2 + 1, 9, 2)
    assert np.abs(got[..., 0] + 1j * got[..., 1] - ref).max() < 1e-12 * np.abs(ref).max()
    back = np.zeros(9 * N)
    _lib.check(g.lib.dmk_fft_backward(g.h, 9, _lib.dptr(out), _lib.dptr(back)))
    assert np.abs(back / N - f.reshape(-1)).max() < 5e-15 * np.log2(N)
    g.close()


@pytest.mark.parametrize("cells", [[64, 144, 2], [144, 64, 2], [128, 72, 1], [72, 128, 2], [192, 48, 1], [28, 320, 1]])
def test_planes_too_large_for_padded_lines_stay_fused(gpu_lib, cells, monkeypatch):
    """planes that fit the two-buffer x-y kernels' LDS with dense lines only"""
    monkeypatch.setenv("DMK_FFT_XY", "1")
    g, _ = _solver(cells)
    assert g.scalar("fft_path")[0] > 0
    g.close()
    test_transforms_against_numpy(gpu_lib, cells, "1", monkeypatch)


@pytest.mark.parametrize("zgz", ["0", "1", "2"])
@pytest.mark.parametrize("cells", [[4, 6, 128], [2, 3, 192], [130, 2, 64], [6, 5, 22]])
def test_gamma_convolution_against_oracle(gpu_lib, oracle, cells, zgz, monkeypatch):
    from damask_amd import _lib, config, workloads
    from damask_amd.config import Numerics
    from damask_amd.grid import GridMechSpectralBasic
    monkeypatch.setenv("DMK_FFT_ZGZ", zgz)
    grid, mat = workloads.polycrystal(cells, 2, 1)
    mat = config.parse_material(mat)
    g, o = GridMechSpectralBasic(grid, mat, Numerics()), oracle.Problem(grid, mat, Numerics())
    N = grid.n_cells
    f = 1e6 * np.random.default_rng(4).random(9 * N)
    aim = np.arange(9.0) * 1e-4
    got, ref = np.zeros(9 * N), np.zeros(9 * N)
    _lib.check(g.lib.dmk_gamma_convolution(g.h, _lib.dptr(f), _lib.dptr(aim), _lib.dptr(got)))
    oracle.lib().orc_gamma_convolution(o.grid, oracle.ptr(f), oracle.ptr(aim), oracle.ptr(ref))
    assert np.abs(got - ref).max() < 1e-12 * np.abs(ref).max()
    g.close()
