"""z lines longer than any segment plan of the z Thomas solves (NCL3 = 500 and
up): the stencil path steps through them, within the 1e-12 of the other FP64
parity tests (Q and CONVH0 against the CPU oracle) and, for the mixed form, the
1e-6 its substep test asks of Q; the Thomas path, and lines that the z transforms'
LDS does not hold, are refused before anything is written."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields
from chapsim1ww_amd import native as nat
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("dims,precision,mode", [((16, 20, 500), "fp64", "auto"), ((16, 20, 500), "fp64", "marching"),
                                                 ((24, 18, 540), "fp64", "rowtile"), ((16, 20, 640), "fp64", "auto"),
                                                 ((32, 18, 640), "mixed", "auto")])
def test_long_z_lines_step_through_the_stencils(dims, precision, mode):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"long z {dims} {precision} {mode}", flush=True)
    hz = np.pi if precision == "fp64" else 10 * np.pi   # cells of the mixed form's proportions
    g, og = ChannelGrid(*dims, hz=hz), O.OracleGrid(*dims, hz=hz)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    st = O.OracleState(og, q, pr, c0)
    dt = 0.4 / st.cfl()
    s = ChannelSolver(g, precision)
    s.set_cn_solver(mode)
    assert s.cn_info(1, dt)["path"] == "stencil"
    s.upload_state(q, pr, c0)
    tol = 1e-12 if precision == "fp64" else 1e-6
    for ns in (0, 1, 2, 3):
        if s.cn_info(ns, dt)["path"] == "thomas":   # NS = 0 at NCL3 = 640: 17 wide
            with pytest.raises(nat.ChsError, match="NCL3"):
                s.solverrk3_mom_tg(ns, dt)
            continue
        st.substep(ns, dt)
        s.solverrk3_mom_tg(ns, dt)
        qg, _, cg = s.download_state()
        assert _rel(qg, st.q) < tol, (ns, _rel(qg, st.q))
        if precision == "fp64":
            assert _rel(cg, st.convh0) < tol, (ns, _rel(cg, st.convh0))
    s.close()


@pytest.mark.parametrize("dims,mode", [((16, 20, 500), "thomas"), ((16, 20, 1080), "auto"),
                                       ((16, 20, 1080), "marching")])
def test_refused_z_lines_leave_the_state(dims, mode):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"refused z {dims} {mode}", flush=True)
    g = ChannelGrid(*dims)
    state = fields.init_tg_fields(g, seed=3)
    s = ChannelSolver(g)
    s.upload_state(*state)
    dt = 0.4 / s.cfl()
    s.set_cn_solver(mode)
    before = s.download_state()
    with pytest.raises(nat.ChsError, match="NCL3"):
        s.solverrk3_mom_tg(1, dt)
    for a, b in zip(before, s.download_state()):
        assert np.array_equal(a, b)
    s.close()
