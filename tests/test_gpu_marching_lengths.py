"""The y-marching kernels on x lengths that fill no whole waves and are no
powers of two (threads past the block's last cell repeat it) and, for the
energy equation, beyond 256 (two k rows per block): the tg substep and the
heated substep against the CPU oracle, within the 1e-12 of the other parity
tests, the thermal fields of the first substep bit for bit.  The tg kernel's
outputs are CONVH0 and, through the line solves, Q; the pressure, whose
round-off the projection divides by the time step, is left to the tests of the
solve and the update."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields, props
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MAP = {"rhoh": "rhoh", "h": "enthalpy", "T": "temperature", "rho": "density", "rho0": "density0",
       "rho1": "density1", "mu": "viscosity", "mu0": "viscosity0", "kap": "thermcondt", "rhs0": "rhs_energy0",
       "g": "g", "g0": "g0", "wallflux": "wallflux", "q": "q", "pr": "pr", "drhodtp": "drhodtp", "divu": "divu",
       "rho_stg": "rho_stg", "mu_stg": "mu_stg", "explt0": "explt0", "drhoi_stg": "drhoi_stg"}


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


@pytest.mark.parametrize("dims", [(24, 40, 20), (40, 33, 24), (72, 20, 32), (120, 24, 20), (200, 18, 20),
                                  (216, 40, 36), (240, 17, 64)])
def test_tg_marching_lengths(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"tg marching {dims}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    st = O.OracleState(og, q, pr, c0)
    dt = 0.4 / st.cfl()
    s = ChannelSolver(g)
    s.set_cn_solver("marching")
    assert s.cn_info(1, dt)["path"] == "stencil"
    s.upload_state(q, pr, c0)
    for ns in (0, 1, 2, 3):
        st.substep(ns, dt)
        s.solverrk3_mom_tg(ns, dt)
        qg, _, cg = s.download_state()
        assert _rel(qg, st.q) < 1e-12 and _rel(cg, st.convh0) < 1e-12, (ns, _rel(qg, st.q), _rel(cg, st.convh0))
    s.close()


@pytest.mark.parametrize("dims", [(18, 12, 8), (32, 9, 8), (36, 20, 12), (50, 13, 16), (90, 12, 8), (120, 17, 12),
                                  (200, 12, 8), (250, 10, 8), (288, 12, 6), (450, 9, 8), (512, 10, 8)])
def test_heated_marching_lengths(dims):
    from chapsim1ww_amd.heated import HeatedChannel
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"heated marching {dims}", flush=True)
    sc = props.scale_table(props.synthetic_table())
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    kw = dict(thermal=1, gravdir=1, f_a=-0.05)
    st, tab, n = O.io_case(og, sc, seed=sum(dims))
    s, pt = ChannelSolver(g), props.PropertyTable(sc)
    s.set_cn_solver("marching")
    hc = HeatedChannel(s, pt, **kw)
    hc.upload({MAP[k]: v for k, v in st.items()})
    io = O.OracleIO(og, st, **kw)
    pr_scale = np.abs(st["pr"]).max()
    for ns in (1, 2, 3):
        O.energy_substep(og, st, tab, n, ns, 1e-3, 1.0 / 2800.0, O.rhoh_max(sc))
        io.prepare(ns)
        io.substep(ns, 1e-3)
        hc.substep(ns, 1e-3, 1.0 / 2800.0)
        got = hc.download()
        if ns == 1:
            for k in ("rhoh", "h", "T", "rho", "mu", "kap", "rhs0"):
                assert np.array_equal(got[MAP[k]], st[k]), k
        for k in ("g", "g0", "explt0", "divu", "q", "rho_stg", "mu_stg", "rho", "T", "h", "rhs0"):
            assert _rel(got[MAP[k]], st[k]) < 1e-12, (ns, k, _rel(got[MAP[k]], st[k]))
        pr_scale = max(pr_scale, np.abs(st["pr"]).max())
        assert np.abs(got["pr"] - st["pr"]).max() < 1e-12 * pr_scale, ns
    pt.close()
    s.close()
