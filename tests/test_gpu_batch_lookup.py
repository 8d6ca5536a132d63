"""The lanes' search for a tile's instance and the per-solver lists, at the
batch sizes where the search takes another round (64 first tiles a load) and
for batches of one solver, of both, and with one instance of the other."""
import numpy as np
import pytest

from helpers import OracleGrid, load_pkg
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,mix", [(2, "alternate"), (3, "one"), (63, "alternate"),
                                   (64, "single"), (65, "single"), (65, "one"),
                                   (129, "alternate"), (130, "single")])
def test_every_instance_of_a_batch_matches_oracle(n, mix):
    pkg = load_pkg()
    rng = np.random.default_rng(n)
    descs, states = [], []
    for k in range(n):
        nx, ny = int(rng.integers(2, 70)), int(rng.integers(2, 12))
        hlle = {"alternate": k % 2, "single": 0, "one": k == n // 2}[mix]
        descs.append(desc(nx, ny, "hlle" if hlle else "roe", (4, 4, 4, 4)))
        states.append(state(nx, ny, 1000 * n + k))
    g = pkg.Grid(descs)
    for k, s in enumerate(states):
        g.upload(k, *s)
        g.set_clock(k, 1e-5 * (1 + k % 3), 0.0, 1)
    g.set_bvals()
    g.set_limits(1e30, -1)
    g.run(2)
    for k, (d, s) in enumerate(zip(descs, states)):
        ora = OracleGrid(d)
        ora.put(*s)
        ora.set_bvals()
        ora.set_time(1e-5 * (1 + k % 3), 0.0, 1)
        for _ in range(2):
            ora.step(1e30)
        assert g.clock(k) == ora.clock(), (n, mix, k)
        for a, b in zip(g.download(k), ora.get()):
            assert np.array_equal(a, b), (n, mix, k, d)
    g.close()
