"""Work of a handle that its caller has captured and replays: the next
main-loop step starts itself, whatever the replay left in the clock."""
import pytest
import torch  # before libathmi.so: torch's HIP runtime serves the process

from test_gpu_fused_ghosts import start

pytestmark = pytest.mark.gpu


def captured_integrate(g, stream):
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        g.integrate()
    return graph


@pytest.mark.parametrize("limit", ["nlim", "tlim", "tpause"])
def test_step_after_a_replayed_integrate_keeps_the_limits(limit):
    """integrate leaves an unconditional start in the clock: a step replayed
    from the handle's own graph after it must not take it for its own."""
    ora, g = start(40, 24, (4, 4, 4, 4), "roe")
    stream = torch.cuda.Stream()
    g.set_stream(stream.cuda_stream)
    g.step()  # makes the step graph
    ora.step(1e30)
    graph = captured_integrate(g, stream)
    dt, t, n = g.clock(0)
    tlim = t + 1.5 * dt if limit == "tlim" else 1e30
    g.set_limits(tlim, n + 1 if limit == "nlim" else -1)
    g.set_pause(t + dt if limit == "tpause" else float("inf"))
    g.step()  # consumes the start that the host's writes asked for
    ora.step(tlim)
    assert g.clock(0) == ora.clock()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        ora.integrate()
        g.set_bvals()
        ora.set_bvals()
        g.step()  # at its limit (nlim, tpause), or clamped to it (tlim)
        if limit == "tlim" and ora.clock()[1] < tlim:
            ora.step(tlim)
        assert g.clock(0) == ora.clock()
    for a, b in zip(g.download(0), ora.get()):
        assert (a == b).all()
    g.close()
