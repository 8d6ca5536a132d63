"""new_dt's maximum where a cell's inverse time step is not a number (a run told
to go on after a non-finite state): such cells are left out, whatever tile,
lane or march they fall in, and every other cell counts. The expected dt is
formed from the state the step produced, cell by cell as new_dt.c:35-90."""
import numpy as np
import pytest

from helpers import load_pkg
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu


def max_inverse_dt(d, gas):
    u = gas[4:-4, 4:-4]
    dx1 = (d["x1max"] - d["x1min"]) / d["nx1"]
    dx2 = (d["x2max"] - d["x2min"]) / d["nx2"]
    with np.errstate(all="ignore"):
        di = 1.0 / u[..., 0]
        v1, v2, v3 = u[..., 1] * di, u[..., 2] * di, u[..., 3] * di
        qsq = v1 * v1 + v2 * v2 + v3 * v3
        p = (d["gamma"] - 1.0) * (u[..., 4] - 0.5 * u[..., 0] * qsq)
        p = np.where(p > 1e-20, p, 1e-20)
        a = np.sqrt(d["gamma"] * p * di)
        m = (np.abs(v1) + a) / dx1
        m2 = (np.abs(v2) + a) / dx2
        m = np.where(m > m2, m, m2)
    assert np.isnan(m).any() and not np.isnan(m).all()
    return np.nanmax(m)


# a 64 x 8 tile and its edges; the corrector-and-final march of each solver
@pytest.mark.parametrize("nx,ny,flux", [(64, 40, "roe"), (130, 36, "hlle"), (1301, 1001, "hlle"),
                                        (1985, 1701, "roe")])
@pytest.mark.parametrize("persist", [0, 1])
def test_cells_without_a_number_are_left_out(nx, ny, flux, persist):
    pkg = load_pkg()
    d = desc(nx, ny, flux, (4, 4, 4, 4))
    s0 = state(nx, ny, nx)
    g = pkg.Grid(d)
    g.set_shape(3, persist)
    g.set_fail_stop(0)
    for n in range(6):
        # the fastest cell of the grid, and a NaN density beyond the step's
        # reach of it: in the same column (n even) or row
        j, i = 4 + (n * 3 + 2) % (ny - 16), 4 + (n * 11 + 1) % (nx - 16)
        gas = s0[0].copy()
        gas[j, i, 1] = 4.0 * gas[j, i, 0]
        gas[j, i, 4] += 8.0 * gas[j, i, 0]
        gas[(j + 8, i) if n % 2 == 0 else (j, i + 8)][0] = np.nan
        g.upload(0, gas, *s0[1:])
        g.set_bvals()
        g.set_clock(0, 1e-6, 0.0, 1)
        g.set_limits(1e30, -1)
        g.run(1)
        want = max_inverse_dt(d, g.download(0)[0])
        # the step's dt doubles at most: let the maximum decide
        assert 2e-6 < 0.4 / want
        g.set_clock(0, 1.0, 0.0, 1)
        g.new_dt()
        assert g.clock(0)[0] == 0.4 / want, (n, "new_dt")
        g.upload(0, gas, *s0[1:])
        g.set_bvals()
        dt = 0.3 / want
        g.set_clock(0, dt, 0.0, 1)
        g.run(1)
        want = max_inverse_dt(d, g.download(0)[0])
        assert g.clock(0)[0] == min(2.0 * dt, 0.4 / want), (n, "step")
    g.close()
