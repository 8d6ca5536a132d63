"""The predictor of grids that leave most of the chip empty (one x2 face per pair
of waves, marches of one face): against the oracle where its x2 tiles end and at
the sizes on both sides of its line (three workgroups per CU), and against the
marches of three faces."""
import numpy as np
import pytest

from helpers import OracleGrid, load_pkg
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu


def tiles(nx, ny):
    return -(-((ny + 4) * (nx + 6) - 3) // 125) + -(-(nx + 4) * (ny + 4) // 64)


@pytest.mark.parametrize("flux", ["roe", "hlle"])
@pytest.mark.parametrize("nx,ny,bc", [(4, 4, (1, 2, 4, 4)), (58, 9, (4, 4, 2, 1)),
                                      (59, 6, (2, 2, 1, 1)), (60, 64, (4, 4, 4, 4)),
                                      (61, 33, (1, 1, 2, 2)), (182, 170, (4, 4, 2, 1)),
                                      (183, 171, (4, 4, 4, 4)),
                                      (193, 181, (2, 1, 4, 4))])
def test_paired_faces_match_oracle_and_marches(nx, ny, bc, flux):
    pkg = load_pkg()
    d = desc(nx, ny, flux, bc)
    s0 = state(nx, ny, nx * 7 + ny)
    ora = OracleGrid(d)
    ora.put(*s0)
    ora.set_bvals()
    ora.set_time(1e-3 / max(nx, ny), 0.0, 1)
    for _ in range(2):
        ora.step(1e30)
    for seg in (1, 3):
        g = pkg.Grid(d)
        g.upload(0, *s0)
        g.set_bvals()
        g.set_clock(0, 1e-3 / max(nx, ny), 0.0, 1)
        g.set_shape(seg, 0)
        g.set_limits(1e30, -1)
        g.run(2)
        got = g.download(0)
        assert g.clock(0) == ora.clock(), (seg, tiles(nx, ny))
        g.close()
        for a, b in zip(got, ora.get()):
            assert np.array_equal(a, b), (seg, tiles(nx, ny))
