"""Time steps of a size of their own each (18 stencils: more than a handle
keeps, so their buffers are reused): every step equal bit for bit to that of a
new handle started from the same state."""
import numpy as np
import pytest

from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(32, 40, 24), (128, 72, 64)])
def test_steps_of_their_own_size(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"time steps of their own size {dims}", flush=True)
    g = ChannelGrid(*dims)
    a = ChannelSolver(g)
    a.upload_state(*fields.init_tg_fields(g, seed=9))
    dt = 0.4 / a.cfl()
    for n in range(6):
        start = a.download_state()
        b = ChannelSolver(g)
        b.upload_state(*start)
        for s in (a, b):
            for ns in (1, 2, 3):
                s.solverrk3_mom_tg(ns, dt)
        for x, y in zip(a.download_state(), b.download_state()):
            assert np.array_equal(x, y), (n, np.abs(x - y).max())
        b.close()
        dt *= 0.93
    a.close()
