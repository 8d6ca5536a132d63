"""set_bvals inside the final update, the main-loop step started by the step
before it, and the allocation-free entry point on scratch that holds an
earlier call's data."""
import ctypes
import itertools

import numpy as np
import pytest
import torch  # before libathmi.so: torch's HIP runtime serves the process

from helpers import OracleGrid, load_pkg
from test_gpu_merged import desc, state

pytestmark = pytest.mark.gpu

BCS = [(4, 4, 4, 4), (1, 1, 1, 1), (2, 2, 2, 2), (1, 2, 4, 4), (4, 4, 2, 1), (2, 1, 1, 2)]
# the smallest that fills from the source's side, cells with ghost images at
# both ends, one row or column short of, at and past a 64 x 8 tile, and a thin
# grid (ghosts that copy ghosts)
SIZES = [(4, 4), (5, 7), (8, 4), (64, 8), (63, 9), (65, 17), (67, 5), (130, 12), (3, 9)]


def start(nx, ny, bc, flux):
    pkg = load_pkg()
    d = desc(nx, ny, flux, bc)
    s0 = state(nx, ny, nx * 100 + ny)
    ora, g = OracleGrid(d), pkg.Grid(d)
    dt = 2e-3 / max(nx, ny)
    ora.put(*s0)
    ora.set_bvals()
    ora.set_time(dt, 0.0, 1)
    g.upload(0, *s0)
    g.set_bvals()
    g.set_clock(0, dt, 0.0, 1)
    g.set_limits(1e30, -1)
    return ora, g


@pytest.mark.parametrize("nx,ny", SIZES)
def test_ghosts_filled_by_the_final_update_match_oracle(nx, ny):
    for bc in BCS:
        ora, g = start(nx, ny, bc, "hlle")
        for rows, fusion in ((8, 1), (4, 0), (16, 1)):
            g.set_final_rows(rows)
            g.set_fusion(fusion)
            g.run(1)
            ora.step(1e30)
            for a, b in zip(g.download(0), ora.get()):
                assert np.array_equal(a, b), (nx, ny, bc, rows, fusion)
            assert g.clock(0) == ora.clock()
        g.close()


@pytest.mark.parametrize("graph", [True, False])
def test_clock_changes_between_steps_take_effect(graph):
    ora, g = start(24, 20, (4, 4, 4, 4), "roe")
    g.use_graph(graph)
    for _ in range(2):
        g.run(2)
        for _ in range(2):
            ora.step(1e30)
        assert g.clock(0) == ora.clock()
    dt, t, n = g.clock(0)
    # a limit inside the next step: dt itself is not clamped before it runs
    g.set_limits(t + 1.25 * dt, -1)
    g.run(1)
    ora.step(t + 1.25 * dt)
    assert g.clock(0) == ora.clock()
    assert g.run(-1) > 0
    ora.run(t + 1.25 * dt, -1)
    assert g.clock(0) == ora.clock() and g.clock(0)[1] >= t + 1.25 * dt
    g.step()  # past the limit: nothing runs
    assert g.clock(0) == ora.clock()
    # a step count limit, a pause, a new dt
    g.set_limits(1e30, ora.clock()[2] + 1)
    g.run(5)
    ora.step(1e30)
    assert g.clock(0) == ora.clock()
    g.set_limits(1e30, -1)
    g.set_pause(ora.clock()[1])
    g.step()
    assert g.clock(0) == ora.clock()
    g.set_pause(float("inf"))
    g.new_dt()
    ora.new_dt()
    g.run(1)
    ora.step(1e30)
    g.integrate()
    ora.integrate()
    g.set_bvals()
    ora.set_bvals()
    g.run(2)
    for _ in range(2):
        ora.step(1e30)
    assert g.clock(0) == ora.clock()
    for a, b in zip(g.download(0), ora.get()):
        assert np.array_equal(a, b)
    g.close()


@pytest.mark.parametrize("flux,bc", itertools.product(["roe", "hlle"], [(4, 4, 4, 4), (1, 2, 2, 1)]))
def test_static_entry_point_reads_no_earlier_scratch(flux, bc):
    pkg = load_pkg()
    for nx, ny in ((120, 33), (58, 64), (3, 2)):
        d = desc(nx, ny, flux, bc)
        g = pkg.Grid(d)
        g.upload(0, *state(nx, ny, 5))
        g.set_bvals()
        g.set_clock(0, 1e-5, 0.0, 1)
        planes, pitch = g.device_state(0)
        ps = (planes[1] - planes[0]) // 8
        c = pkg._Desc(nx, ny, d["x1min"], d["x1max"], d["x2min"], d["x2max"], d["gamma"], 0.4,
                      *bc, pkg.FLUXES[flux], pkg.EXACT)
        nan = torch.full((11 * ps,), float("nan"), dtype=torch.float64, device="cuda")
        out = [torch.full((11 * ps,), float("nan"), dtype=torch.float64, device="cuda")
               for _ in range(2)]
        torch.cuda.synchronize()
        # a NaN state leaves NaN in every scratch plane; then the real one
        for src, dst in ((nan.data_ptr(), out[0]), (planes[0], out[1])):
            pkg._check(pkg.lib().athmi_integrate_static(
                ctypes.byref(c), 1e-5, ctypes.c_void_p(src), ctypes.c_void_p(dst.data_ptr()),
                pitch, ps, None), "athmi_integrate_static")
        torch.cuda.synchronize()
        sy, sx = ny + 8, nx + 8
        got = out[1].cpu().numpy().reshape(11, ps)[:, :sy * pitch].reshape(11, sy, pitch)[:, :, :sx]
        g.integrate()
        gas, b1i, b2i, b3i = g.download(0)
        want = [gas[..., f] for f in range(8)] + [b1i, b2i, b3i]
        for f in range(11):
            assert np.array_equal(got[f], want[f]), (nx, ny, f)
        g.close()


def test_clock_read_between_replays_of_a_captured_step():
    """Steps the caller has captured change the clocks without a call: every
    read still gives the device's."""
    ora, g = start(40, 24, (4, 4, 4, 4), "roe")
    g.use_graph(False)
    stream = torch.cuda.Stream()
    g.set_stream(stream.cuda_stream)
    g.step()
    ora.step(1e30)
    assert g.clock(0) == ora.clock()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        g.step()
    for n in range(4):
        graph.replay()
        torch.cuda.synchronize()
        ora.step(1e30)
        assert g.clock(0) == ora.clock(), n
        for a, b in zip(g.download(0), ora.get()):
            assert np.array_equal(a, b), n
    g.set_limits(1e30, ora.clock()[2] + 1)  # the captured step starts itself
    for _ in range(3):
        graph.replay()
    torch.cuda.synchronize()
    ora.step(1e30)
    assert g.clock(0) == ora.clock()
    g.close()
