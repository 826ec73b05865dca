"""Several threads reading fields of one handle, and one more using the handle's
spectral operators, get what each gets alone, bit for bit."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_fields_read_by_several_threads(gpu_lib):
    from damask_amd import _lib, config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    grid, mat = workloads.polycrystal([16, 16, 17], 5, 3)
    g = GridMechSpectralBasic(grid, config.parse_material(mat))
    N = grid.n_cells
    rng = np.random.default_rng(1)
    F = np.eye(3) + 4e-4 * np.diag([1.0, -0.4, -0.4]) + 2e-4 * rng.standard_normal((N, 3, 3))
    assert g.constitutive(F, 0.5)[4] == 0
    field, aim = 1e6 * rng.random(9 * N), np.arange(9.0) * 1e-4

    def convolution():
        out = np.zeros(9 * N)
        _lib.check(g.lib.dmk_gamma_convolution(g.h, _lib.dptr(field), _lib.dptr(aim), _lib.dptr(out)))
        return out

    reads = {n: (lambda n=n: g.field(n)) for n in ("P", "F_p", "dPdF", "xi_sl", "gamma_sl", "S")}
    reads["convolution"] = convolution
    alone = {n: f() for n, f in reads.items()}
    wrong = []

    def worker(n):
        for _ in range(20):
            if not np.array_equal(reads[n](), alone[n]):
                wrong.append(n)

    threads = [threading.Thread(target=worker, args=(n,)) for n in reads]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    g.close()
