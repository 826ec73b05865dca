"""A lockstep batch with every kernel variant of the stress integration in its
rounds: 12 and 24 systems, Schmid law and non-Schmid terms, quarter powers and
free exponents.  Curves equal the single runs bit for bit."""
import numpy as np
import pytest

from test_gpu_slip_variants import _phase

pytestmark = pytest.mark.gpu

VARIANTS = [("cF", [20.0], [2.25], False), ("cF", [17.3], [2.1], False),
            ("cI", [20.0, 20.0], [2.0, 2.0], False), ("cI", [20.0, 17.3], [2.0, 2.1], False),
            ("cI", [20.0], [2.0], True), ("cI", [20.0], [2.1], True),
            ("cI", [20.0, 20.0], [2.0, 2.0], True), ("cI", [20.0, 20.0], [2.0, 2.1], True)]


def test_all_variants_in_one_round(gpu_lib, monkeypatch):
    from damask_amd import adjoint, batch, config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    monkeypatch.delenv("DMK_LOCKSTEP", raising=False)
    monkeypatch.setenv("DMK_LOCKSTEP_GROUPS", "1")
    items = []
    for k, v in enumerate(VARIANTS):
        grid, mat = workloads.polycrystal([4, 4, 4], 3, 5 + k, phase=_phase(*v))
        items.append((grid, config.parse_material(mat), config.parse_load(workloads.tension_x(1.0, 2))[1][0]))
    b = batch.Batch(items)
    b.tape()
    b.run(threads=len(items), lockstep=True)
    curves = b.curves()
    b.close()
    for (grid, mat, lc), c in zip(items, curves):
        s = GridMechSpectralBasic(grid, mat)
        s.adjoint_tape(2 * lc.N + 16)
        assert s.run_loadcase(lc)["rc"] == 0
        assert np.array_equal(adjoint._P33(s.adjoint_info()["P_av"]), c)
        s.close()


def test_one_grid_shares_its_transforms(gpu_lib, monkeypatch, capfd):
    """RVEs of one grid whose set-ups picked other shapes for the fused transforms run
    them in the same launches of a round; results equal the single runs bit for bit, and
    each handle has its own shapes back."""
    import re

    from damask_amd import adjoint, batch, config, workloads
    from damask_amd.grid import GridMechSpectralBasic
    monkeypatch.delenv("DMK_LOCKSTEP", raising=False)
    monkeypatch.setenv("DMK_LOCKSTEP_GROUPS", "1")
    monkeypatch.setenv("DMK_LOCKSTEP_WAIT_US", "")
    monkeypatch.setenv("DMK_BATCH_TIMING", "1")
    items = []
    for k in range(4):
        grid, mat = workloads.polycrystal([8, 8, 8], 3, 5 + k)
        items.append((grid, config.parse_material(mat), config.parse_load(workloads.tension_x(1.0, 2))[1][0]))
    b = batch.Batch(items)
    for s in b.solvers:
        s.close()
    b.solvers = []
    for (grid, mat, _), force in zip(items, "1212"):
        monkeypatch.setenv("DMK_FFT_XY", force)
        monkeypatch.setenv("DMK_FFT_ZGZ", force)
        b.solvers.append(GridMechSpectralBasic(grid, mat))
    for i, s in enumerate(b.solvers):
        b._h[i] = s.h.value
    paths = [s.scalar("fft_path").tolist() for s in b.solvers]
    assert paths[0][1] != paths[1][1] and paths[0][4] != paths[1][4]
    b.tape()
    b.run(threads=4, lockstep=True)
    curves = b.curves()
    assert [s.scalar("fft_path").tolist() for s in b.solvers] == paths
    per_round = re.search(r"transforms in ([0-9.]+) launches", capfd.readouterr().err)
    assert per_round and float(per_round.group(1)) <= 1.0
    b.close()
    monkeypatch.delenv("DMK_FFT_XY")
    monkeypatch.delenv("DMK_FFT_ZGZ")
    for (grid, mat, lc), c in zip(items, curves):
        s = GridMechSpectralBasic(grid, mat)
        s.adjoint_tape(2 * lc.N + 16)
        assert s.run_loadcase(lc)["rc"] == 0
        assert np.array_equal(adjoint._P33(s.adjoint_info()["P_av"]), c)
        s.close()
