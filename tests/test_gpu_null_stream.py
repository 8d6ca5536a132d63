"""Reads of the clock or the state wait for work on the null stream: a replay
there of steps the caller has captured, and a caller's own kernels on the
planes."""
import pytest
import torch  # before libathmi.so: torch's HIP runtime serves the process

from test_gpu_fused_ghosts import start

pytestmark = pytest.mark.gpu


def test_reads_wait_for_a_replay_on_the_null_stream():
    ora, g = start(48, 32, (4, 4, 4, 4), "hlle")
    g.use_graph(False)
    stream = torch.cuda.Stream()
    g.set_stream(stream.cuda_stream)
    g.step()
    ora.step(1e30)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        g.step()
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    for read in ("clock", "download", "clock"):
        for _ in range(20):  # keeps the null stream busy for some milliseconds
            a = torch.nn.functional.normalize(a @ a)
        graph.replay()  # torch's current stream: the null stream
        ora.step(1e30)
        if read == "clock":
            assert g.clock(0) == ora.clock()
        else:
            for x, y in zip(g.download(0), ora.get()):
                assert (x == y).all()
    g.close()


def test_download_waits_for_the_callers_kernels_on_the_null_stream():
    ora, g = start(48, 32, (4, 4, 4, 4), "hlle")
    ptr, pitch = g.device_state(0)
    sy, sx = g.shape(0)

    class Energy:
        __cuda_array_interface__ = {"shape": (sy, sx), "strides": (pitch * 8, 8), "typestr": "<f8",
                                    "data": (ptr[4], False), "version": 3}

    energy = torch.as_tensor(Energy(), device="cuda")
    a = torch.randn(4096, 4096, device="cuda")
    torch.cuda.synchronize()
    want = ora.get()[0].copy()
    for n in range(3):
        for _ in range(20):
            a = torch.nn.functional.normalize(a @ a)
        energy.add_(0.5)
        want[..., 4] += 0.5
        assert (g.download(0)[0] == want).all(), n
    g.close()
