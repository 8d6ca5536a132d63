"""A thread that polls the clock while another steps the grid: every read that
follows a step sees it, and the polled step counts never go back."""
import threading

import pytest

from test_gpu_fused_ghosts import start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [400])
def test_clock_polled_from_another_thread(steps):
    ora, g = start(24, 16, (4, 4, 4, 4), "hlle")
    g.step()  # makes the step graph: a stream under capture cannot be waited for
    ora.step(1e30)
    n0 = g.clock(0)[2]
    done = threading.Event()
    polled = []

    def poll():
        while not done.is_set():
            polled.append(g.clock(0)[2])

    t = threading.Thread(target=poll)
    t.start()
    try:
        for n in range(1, steps + 1):
            g.step()
            ora.step(1e30)
            assert g.clock(0)[2] == n0 + n
    finally:
        done.set()
        t.join()
    assert polled == sorted(polled)
    assert g.clock(0) == ora.clock()
    for a, b in zip(g.download(0), ora.get()):
        assert (a == b).all()
    g.close()
