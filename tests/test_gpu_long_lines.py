"""The marching RHS kernel on x lines beyond 256 values (two k rows per block,
the x-solve rows in the ring): lengths that fill no whole waves, chunks of one
and of several, every width of the x window; the tg substep against the CPU
oracle within the 1e-12 of the other parity tests."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("nflow", [1, 3])
@pytest.mark.parametrize("dims,f", [((288, 20, 20), 0.4), ((360, 17, 24), 0.4), ((512, 18, 20), 0.4),
                                    ((400, 40, 36), 0.4), ((512, 24, 32), 4.0), ((320, 24, 32), 0.02)])
def test_tg_long_lines(dims, f, nflow):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"tg long lines {dims} {f} nflow={nflow}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=5)
    st = O.OracleState(og, q, pr, c0)
    dt = f / st.cfl()
    s = ChannelSolver(g, "fp64", nflow=nflow)
    s.set_cn_solver("marching")
    assert s.cn_info(1, dt)["path"] == "stencil", s.cn_info(1, dt)
    s.upload_state(q, pr, c0)
    for ns in (0, 1, 2):
        st.substep(ns, dt, 1, nflow, 0.0)
        s.solverrk3_mom_tg(ns, dt)
        qg, _, cg = s.download_state()
        assert _rel(qg, st.q) < 1e-12 and _rel(cg, st.convh0) < 1e-12, (ns, _rel(qg, st.q), _rel(cg, st.convh0))
    s.close()
