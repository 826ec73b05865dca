"""Dot products of a residual evaluation where jobs share a block or not.

Sizes: less than a chunk of 2048 values; chunks enough for one, a few and the most
jobs of a block, 8 (the rule takes chunks x jobs / 1024 jobs a block), with last blocks of fewer.
Values against sums in long double: a chunk's products are summed by 256 threads of 8
values, then in a tree, then the chunks 256 at a time and in a tree, so a sum of n
carries at most 8 + 8 + n / (2048 * 256) + 8 + 2 roundings of the products' absolute sum.

In a run the products steer the iteration only: its converged P equals that of a run without
acceleration (Richardson) within what both leave of the divergence,
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


# (values, vectors, jobs as (x, y, mode)), jobs a block by the rule: 1 1 2 3 8 8
def _against(x, ys, mode=0):
    return [(x, y, mode) for y in ys]


JOBS = [(1, 2, [(0, 1, 0), (1, 1, 0), (0, 1, 1)]),
        (2047, 3, [(0, 1, 0), (0, 2, 1), (2, 2, 0), (1, 2, 0), (1, 1, 1)]),
        (2048 * 300 + 5, 4, _against(0, (1, 2, 3)) + _against(2, (1, 3), 1) + [(3, 3, 0), (3, 0, 0)]),
        (2048 * 341 + 2047, 3, _against(0, (0, 1, 2)) + _against(1, (0, 1, 2), 1) + _against(2, (2, 1, 0))
         + [(0, 2, 1)]),
        (2048 * 700 + 3, 4, _against(0, (1, 2, 3, 0)) * 2 + _against(1, (0, 2), 1) + _against(2, (2, 1, 3))),
        (2048 * 1200 + 1, 3, [(0, 1, 0), (1, 0, 0), (1, 1, 0), (2, 1, 1), (2, 0, 0), (0, 0, 0), (2, 2, 0)])]


@pytest.mark.parametrize("case", range(len(JOBS)))
def test_values(gpu_lib, case):
    from damask_amd import _lib
    n, n_vec, jobs = JOBS[case]
    v = np.random.default_rng(case).standard_normal((n_vec, n))
    x, y, mode = (np.array([j[k] for j in jobs], np.int32) for k in range(3))
    out = np.zeros(len(jobs))
    _lib.check(gpu_lib.dmk_dot_products(_lib.dptr(v.reshape(-1)), n, n_vec, _lib.iptr(x), _lib.iptr(y), _lib.iptr(mode),
                                        len(jobs), _lib.dptr(out)), "dmk_dot_products")
    L = v.astype(np.longdouble)
    for (a, b, m), got in zip(jobs, out):
        terms = L[a] * L[b] if m == 0 else (L[b] - L[a]) ** 2
        roundings = 26 + n / (2048 * 256) + (2 if m else 0)      # mode 1: the difference's, squared
        assert abs(got - terms.sum()) <= roundings * 2.0**-53 * np.abs(terms).sum(), (a, b, m)
