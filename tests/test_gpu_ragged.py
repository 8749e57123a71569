"""Substeps of the tg channel on grids whose sizes no tile or chunk divides,
against the CPU oracle: z lines of any length through the z window (a shorter
last chunk among them), the shortest z lines of that path and one below it.  Tolerance: the 1e-12 of the other FP64 parity
tests (each field relative to its largest value, after every substep)."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("dims,path", [((32, 40, 32), "stencil"), ((64, 20, 36), "stencil"), ((24, 33, 100), "stencil"),
                                       ((48, 17, 60), "stencil"), ((64, 70, 144), "stencil"), ((32, 40, 20), "stencil"),
                                       ((64, 64, 24), "stencil"), ((32, 40, 16), "thomas")])
@pytest.mark.parametrize("nflow,drive", [(1, 1), (3, 2)])
def test_substep_any_z_length(dims, path, nflow, drive):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"substep {dims} nflow={nflow} drive={drive}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=5)
    cfgv = 0.02 if drive == 2 else 0.0
    st = O.OracleState(og, q, pr, c0)
    dt = 0.4 / st.cfl()
    s = ChannelSolver(g, "fp64", flowdrvtp=drive, nflow=nflow, cfgv=cfgv)
    assert s.cn_info(1, dt)["path"] == path
    s.upload_state(q, pr, c0)
    for ns in (0, 1, 2, 3):
        st.substep(ns, dt, drive, nflow, cfgv)
        s.solverrk3_mom_tg(ns, dt)
        for name, a, b in zip(("Q", "PR", "CONVH0"), s.download_state(), (st.q, st.pr, st.convh0)):
            assert _rel(a, b) < 1e-12, (ns, name, _rel(a, b))
    s.close()


def test_mixed_form_keeps_fp64_stencils_off_64():
    """The mixed form's FP32 stencils need NCL3 a multiple of 64; elsewhere its
    momentum part stays FP64: CONVH0 of the first substep equals the FP64
    form's bit for bit."""
    g = ChannelGrid(64, 48, 72)
    q, pr, c0 = fields.init_tg_fields(g, seed=9)
    from chapsim1ww_amd.solver import ChannelSolver
    out = []
    for prec in ("fp64", "mixed"):
        s = ChannelSolver(g, prec)
        s.upload_state(q, pr, c0)
        s.solverrk3_mom_tg(1, 0.4 / s.cfl())
        out.append(s.download_state()[2])
        s.close()
    assert np.array_equal(*out)
