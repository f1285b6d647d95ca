"""The launch shape an ensemble gets by itself, on both sides of its rule's
lines (512, 4096 and 8192 row tiles; a mean fan-in of 64, 384, 512, 1024 and
8000; FP32 rows of a multiple of 2048), against the shape of one wavefront a
row tile.

A row's sum is the same products in another grouping: FP32 accumulation over
up to 8192 terms of size 1/sqrt(8192) differs by about sqrt(8192) half units
in the last place of a sum near 1, 3e-6, and less than 1e-5 of the largest
state.
"""

import numpy as np
import pytest

from synaptogenesis_amd.ensemble import RateEnsemble

# widths, precision, the shape expected
SHAPES = [([[40, 4096, 4096]], "bf16", (1, 8)),      # 512 row tiles
          ([[40, 4096, 4097]], "bf16", (2, 4)),      # 513, long rows
          ([[33, 8192, 16], [17, 5, 3]], "bf16", (2, 2)),   # 515, short rows
          ([[31, 17, 3]], "bf16", (2, 1)),           # fan-ins of one load
          ([[65, 17, 3]], "bf16", (1, 8)),
          ([[64, 65, 33]] * 130, "bf16", (2, 2)),    # 1040, mean fan-in 76
          ([[60, 64, 64]] * 130, "bf16", (4, 1)),    # 1040, 64
          ([[100, 100, 100]] * 586, "bf16", (4, 1)),     # 8204, 128
          ([[100, 100, 100]] * 585, "bf16", (2, 2)),     # 8190
          ([[400, 400, 400]] * 82, "bf16", (4, 1)),      # 4100, 416
          ([[400, 400, 400]] * 81, "bf16", (2, 2)),      # 4050
          ([[8192, 8192, 16], [8192, 16, 1]], "bf16", (4, 4)),
          ([[100, 33, 65], [7, 1, 2]], "fp32", (8, 1)),
          ([[100, 100, 100]] * 11, "fp32", (4, 1)),      # 550 row groups
          ([[2048, 2048, 2]], "fp32", (4, 1)),       # 513
          ([[2048, 2040, 8]], "fp32", (8, 1)),       # 512
          ([[4096, 100, 4000]], "fp32", (8, 1)),     # even rows in the minority
          ([[4096, 300, 10]], "fp32", (16, 1))]


@pytest.mark.gpu
@pytest.mark.parametrize("widths,precision,shape", SHAPES)
def test_default_shape(widths, precision, shape):
    states = []
    for tile in (None, (4, 1)):
        e = RateEnsemble(widths, precision, leak=0.3)
        if tile is None:
            assert e.tile == shape
        else:
            e.set_tile(*tile)
        e.run(5)
        states.append([e.state(i, k) for i in range(len(widths))
                       for k in (1, 2)])
        e.close()
    for a, b in zip(*states):
        assert np.abs(a - b).max() <= 1e-5 * max(1e-3, np.abs(b).max())


@pytest.mark.gpu
def test_reads_follow_every_change():
    """Enough reads bring the whole state over at once; runs, writes, timing
    and tuning in between must show, whichever way a read is served."""
    widths = [[40, 70, 33], [5, 64, 100], [17, 3, 9]]
    e = RateEnsemble(widths, "bf16", leak=0.5)
    f = RateEnsemble(widths, "bf16", leak=0.5)

    def every(a):
        return [a.state(i, k) for i in range(3) for k in range(3)]

    def alone():
        # a single read a run: never from the mirror
        out = []
        for i in range(3):
            for k in range(3):
                f.set_state(0, 0, f.state(0, 0))
                out.append(f.state(i, k))
        return out

    for step in range(4):
        for a in (e, f):
            a.run(1 + step, graph=step % 2 == 0)
        for _ in range(3):
            for x, y in zip(every(e), alone()):
                assert np.array_equal(x, y)
        new = np.linspace(0, 1, 70, dtype=np.float32) * step
        for a in (e, f):
            a.set_state(0, 1, new)
        assert np.array_equal(every(e)[1], new)
        e.autotune(1)
        f.set_tile(*e.tile)
        assert np.array_equal(every(e)[1], new)
    e.close()
    f.close()


@pytest.mark.gpu
def test_reads_after_a_callers_graph():
    """Runs recorded into a caller's graph change the state at every replay,
    unseen by the ensemble: however many states were read before, each read
    shows the state as it is."""
    import torch
    widths = [[40, 70, 33], [5, 64, 100], [17, 3, 9]]
    e = RateEnsemble(widths, "bf16", leak=0.5)
    f = RateEnsemble(widths, "bf16", leak=0.5)

    def every(a):
        return [a.state(i, k) for i in range(3) for k in range(3)]

    for _ in range(3):
        every(e)                # the whole state on the host
    graph = torch.cuda.CUDAGraph()
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        e.run(2, graph=False,
              stream=torch.cuda.current_stream().cuda_stream)
    for replay in range(4):
        graph.replay()
        torch.cuda.synchronize()
        f.run(2, graph=False)
        for _ in range(3):
            for x, y in zip(every(e), every(f)):
                assert np.array_equal(x, y)
        if replay == 1:         # the program's own steps in between
            e.run(2)
            f.run(2)
    e.close()
    f.close()


@pytest.mark.gpu
def test_read_without_a_buffer_is_refused():
    """A null buffer is an error, also where the read would be served from
    the host copy of the whole state."""
    e = RateEnsemble([[40, 70, 33]], "bf16")
    for _ in range(20):
        e.state(0, 1)
    assert e.lib.sg_ens_read_state(e.handle, 0, 1, None) != 0
    assert e.state(0, 1).shape == (70,)
    e.close()
