"""The z and y window solves in one pass (mode 'marching'): k tiles and i tiles
that the grid does not fill, pieces that span several components, window
widths 4, 8 and 12 of the y solve, against the CPU oracle within the 1e-12 of
the other parity tests; the mixed form against its two separate windows, from
which only FP32 roundings of an increment (6e-8 of it) could differ."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


GRIDS = [(24, 18, 20), (72, 33, 36), (64, 40, 32), (200, 20, 100), (96, 65, 48)]
# the widest y window needs rows close together at the wall
FINE = [(24, 66, 20), (72, 90, 36), (200, 80, 36), (96, 128, 24)]


@pytest.mark.parametrize("dims,ky", [(d, k) for k in ((1, 4), (5, 8)) for d in GRIDS] + [(d, (9, 12)) for d in FINE])
def test_zy_window(dims, ky):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"zy window {dims} ky {ky}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    st = O.OracleState(og, q, pr, c0)
    s = ChannelSolver(g)
    s.set_cn_solver("marching")
    dt = 4.0 / st.cfl()
    while s.cn_info(1, dt)["ky"] > ky[1]:
        dt *= 0.7
    info = s.cn_info(1, dt)
    assert info["path"] == "stencil" and info["kz"] <= 8 and ky[0] <= info["ky"] <= ky[1], info
    s.upload_state(q, pr, c0)
    for ns in (0, 1):
        st.substep(ns, dt)
        s.solverrk3_mom_tg(ns, dt)
        qg, _, cg = s.download_state()
        assert _rel(qg, st.q) < 1e-12 and _rel(cg, st.convh0) < 1e-12, (ns, info, _rel(qg, st.q))
    s.close()


@pytest.mark.parametrize("dims", [(48, 20, 64), (64, 40, 128)])
def test_zy_window_mixed(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"zy window mixed {dims}", flush=True)
    g = ChannelGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    out = []
    for mode in ("auto", "marching"):
        s = ChannelSolver(g, "mixed")
        s.set_cn_solver(mode)
        s.upload_state(q, pr, c0)
        dt = 0.4 / s.cfl()
        for ns in (0, 1, 2):
            s.solverrk3_mom_tg(ns, dt)
        out.append(s.download_state()[0])
        s.close()
    assert _rel(out[1], out[0]) < 1e-8, _rel(out[1], out[0])
