"""Both sweeps' predictors in one launch, both corrector parts in one launch:
the merged kernels against the oracle where their tiles end -- one face short
of, at and past an x1 tile (125 faces) and an x2 chunk (64 columns), an odd
number of x2 tiles (the last workgroup's second wave has none), the smallest
grids -- and against the separate launches of a persistent grid."""
import numpy as np
import pytest

from helpers import OracleGrid, load_pkg

pytestmark = pytest.mark.gpu

SIZES = [(2, 2), (3, 5), (57, 4), (58, 7), (59, 6), (120, 9), (121, 5), (122, 3), (186, 13),
         (246, 4), (247, 11), (64, 65)]


def state(nx, ny, seed):
    rng = np.random.default_rng(seed)
    gas = rng.uniform(-0.3, 0.3, (ny + 8, nx + 8, 8))
    gas[..., 0] = rng.uniform(0.8, 1.4, (ny + 8, nx + 8))
    gas[..., 4] = rng.uniform(2.0, 3.0, (ny + 8, nx + 8))
    return (gas, *rng.uniform(-0.3, 0.3, (3, ny + 8, nx + 8)))


def desc(nx, ny, flux, bc):
    return dict(nx1=nx, nx2=ny, x1min=-0.5, x1max=0.5, x2min=-0.5 * ny / nx, x2max=0.5 * ny / nx,
                gamma=1.6666666666666667, cour_no=0.4, bc=bc, flux=flux)


@pytest.mark.parametrize("flux", ["roe", "hlle"])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_merged_sweeps_match_oracle_and_separate_launches(nx, ny, flux):
    pkg = load_pkg()
    d = desc(nx, ny, flux, (4, 4, 1, 2) if nx % 2 else (2, 1, 4, 4))
    s0 = state(nx, ny, nx * 1000 + ny)
    ora = OracleGrid(d)
    ora.put(*s0)
    ora.set_bvals()
    ora.set_time(2e-3 / max(nx, ny), 0.0, 1)
    for _ in range(2):
        ora.step(1e30)
    want = ora.get()
    for seg, persist in ((1, 0), (3, 0), (16, 0), (3, 1)):
        g = pkg.Grid(d)
        g.upload(0, *s0)
        g.set_bvals()
        g.set_clock(0, 2e-3 / max(nx, ny), 0.0, 1)
        g.set_shape(seg, persist)
        g.set_limits(1e30, -1)
        g.run(2)
        got = g.download(0)
        g.close()
        for a, b in zip(got, want):
            assert np.array_equal(a, b), (nx, ny, flux, seg, persist)
