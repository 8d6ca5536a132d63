"""The march that holds the corrector, its corners and the final update: taken
by the solver whose marches fill the chip's rounds of waves well. The ensembles
are sized (for 256 CUs) so that marches of 8 rows are one full round; they hold
grids that end one cell short of, at and past a strip of 62 columns and a
march and every boundary type, with none, a few or as many grids of the other
solver beside them, and each grid is checked against the oracle. Large grids,
with marches of 7 to 14 rows, are checked against the separate launches of a
persistent grid."""
import numpy as np
import pytest

from helpers import OracleGrid, load_pkg
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu

EDGES = [(61, 7), (62, 8), (63, 9), (124, 16), (125, 17), (123, 15), (4, 4), (187, 25), (70, 4),
         (5, 32)]
BCS = [(4, 4, 4, 4), (1, 2, 4, 4), (4, 4, 2, 1), (1, 1, 2, 2), (2, 1, 1, 2)]
FILLER = (248, 40)  # 20 marches of 8 rows
FILLERS = {"hlle": 142, "roe": 96}  # twelve and eight waves per CU with the edges


@pytest.mark.parametrize("main,others", [("hlle", 0), ("hlle", 3), ("hlle", 100), ("roe", 0),
                                         ("roe", 3), ("roe", 150)])
def test_ensemble_matches_oracle(main, others):
    pkg = load_pkg()
    other = "roe" if main == "hlle" else "hlle"
    kinds = [(n, b, main) for k, n in enumerate(EDGES) for b in (BCS[k % 5], BCS[(k + 2) % 5])]
    of = list(range(len(kinds))) + [len(kinds)] * FILLERS[main]
    kinds.append((FILLER, BCS[1], main))
    of += [len(kinds)] * others
    kinds.append((FILLER, BCS[4], other))
    descs = [desc(*kinds[q][0], kinds[q][2], kinds[q][1]) for q in of]
    want = []
    for q, ((nx, ny), bc, flux) in enumerate(kinds):
        ora = OracleGrid(desc(nx, ny, flux, bc))
        ora.put(*state(nx, ny, q))
        ora.set_bvals()
        ora.set_time(1e-3 / max(nx, ny), 0.0, 1)
        for _ in range(3):
            ora.step(1e30)
        want.append((ora.get(), ora.clock()))
    g = pkg.Grid(descs)
    for k, q in enumerate(of):
        g.upload(k, *state(*kinds[q][0], q))
    g.set_bvals()
    for k, q in enumerate(of):
        g.set_clock(k, 1e-3 / max(kinds[q][0]), 0.0, 1)
    g.set_limits(1e30, -1)
    g.run(3)
    for k, q in enumerate(of):
        got = g.download(k)
        for a, b in zip(got, want[q][0]):
            assert np.array_equal(a, b), (k, kinds[q])
        assert g.clock(k) == want[q][1], (k, kinds[q])
    g.close()


# fast: the two paths contract different multiplications into FMAs, a few
# hundred roundings a step of at most 2^-53 of the largest term each
@pytest.mark.parametrize("variant,tol", [("exact", 0.0), ("fast", 1e-11)])
@pytest.mark.parametrize("nx,ny,flux,bc", [(1301, 1001, "hlle", (4, 4, 1, 2)),
                                           (1240, 1040, "hlle", (2, 1, 4, 4)),
                                           (1985, 1701, "roe", (1, 2, 4, 4))])
def test_large_grid_matches_separate_launches(nx, ny, flux, bc, variant, tol):
    pkg = load_pkg()
    d = desc(nx, ny, flux, bc)
    s0 = state(nx, ny, nx)
    outs = []
    for persist in (0, 1):
        g = pkg.Grid(d, variant=variant)
        g.upload(0, *s0)
        g.set_bvals()
        g.set_clock(0, 1e-3 / max(nx, ny), 0.0, 1)
        g.set_shape(3, persist)
        g.set_limits(1e30, -1)
        g.run(3)
        outs.append((g.download(0), g.clock(0)))
        g.close()
    for a, b in zip(outs[0][0], outs[1][0]):
        assert np.abs(a - b).max() <= tol * np.abs(b).max()
    assert abs(outs[0][1][0] - outs[1][1][0]) <= tol * outs[1][1][0]


# integrate_2d alone: the march leaves the ghosts as they were
@pytest.mark.parametrize("nx,ny,flux,bc", [(1301, 1001, "hlle", (4, 4, 1, 2)),
                                           (1985, 1701, "roe", (2, 1, 4, 4))])
def test_large_grid_integrate_alone(nx, ny, flux, bc):
    pkg = load_pkg()
    d = desc(nx, ny, flux, bc)
    s0 = state(nx, ny, nx)
    outs = []
    for persist in (0, 1):
        g = pkg.Grid(d)
        g.upload(0, *s0)
        g.set_clock(0, 1e-3 / max(nx, ny), 0.0, 1)
        g.set_shape(3, persist)
        for _ in range(2):
            g.integrate()
        outs.append((g.download(0), g.clock(0)))
        g.close()
    for a, b in zip(outs[0][0], outs[1][0]):
        assert np.array_equal(a, b)
    assert outs[0][1] == outs[1][1]
