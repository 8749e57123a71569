"""Time steps captured in a graph keep their stencils: replays after more step
sizes than a handle keeps, with and without eager steps of the captured size in
between, and step sizes first met inside a capture, all equal bit for bit to the
eager step from the same state (each replay checked, eager work and
synchronisations between them)."""
import numpy as np
import pytest

from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _step(s, dt):
    for ns in (1, 2, 3):
        s.solverrk3_mom_tg(ns, dt)


def _same(s, ref):
    torch.cuda.synchronize()
    return all(np.array_equal(a, b) for a, b in zip(s.download_state(), ref))


def _handle(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    g = ChannelGrid(*dims)
    stream = torch.cuda.Stream()
    s = ChannelSolver(g, stream=stream)
    start = fields.init_tg_fields(g, seed=9)
    s.upload_state(*start)
    return s, stream, start, 0.4 / s.cfl()


@pytest.mark.parametrize("dims", [(32, 40, 24), (64, 40, 64)])
def test_replays_outlive_the_stencil_cache(dims):
    print(f"graph replays {dims}", flush=True)
    s, stream, start, dt = _handle(dims)
    _step(s, dt)
    ref = [a.copy() for a in s.download_state()]
    s.upload_state(*start)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        _step(s, dt)
    d = dt
    for turn in range(4):
        s.upload_state(*start)
        graph.replay()
        assert _same(s, ref), turn
        if turn % 2:   # an eager step of the captured size
            s.upload_state(*start)
            _step(s, dt)
            assert _same(s, ref), turn
        for _ in range(5):   # 15 stencils: more than a handle keeps
            d *= 0.97
            s.upload_state(*start)
            _step(s, d)
        torch.cuda.synchronize()
    s.close()


def test_step_size_first_met_in_a_capture():
    print("graph with a new step size", flush=True)
    s, stream, start, dt = _handle((64, 40, 64))
    _step(s, dt)   # the kernels loaded, their attributes set
    new = 0.9 * dt
    s.upload_state(*start)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="relaxed"):
        _step(s, new)
    from chapsim1ww_amd.solver import ChannelSolver
    b = ChannelSolver(s.grid)
    b.upload_state(*start)
    _step(b, new)
    ref = [a.copy() for a in b.download_state()]
    b.close()
    s.upload_state(*start)
    _step(s, new)   # eager before the first replay
    assert _same(s, ref)
    for _ in range(3):
        s.upload_state(*start)
        graph.replay()
        assert _same(s, ref)
        _step(s, 0.8 * dt)
    s.close()
