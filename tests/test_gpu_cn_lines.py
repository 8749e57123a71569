"""The line solves of the heated channel's RK-CN branch and the batched cyclic
solver on lengths where the segment plan changes: segments of 8, 12 and 4
rows, one or two segments per line, y lines that no segment divides, long
lines (few per block), more lines than fill the last block.  G and G0 after
two substeps within 1e-12 of the CPU oracle (the bound of the heated parity
tests; the solves are diagonally dominant, so their own round-off is a few
eps).  A grid that refused a length still refuses it."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import props
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

MAP = {"rhoh": "rhoh", "h": "enthalpy", "T": "temperature", "rho": "density", "rho0": "density0",
       "rho1": "density1", "mu": "viscosity", "mu0": "viscosity0", "kap": "thermcondt", "rhs0": "rhs_energy0",
       "g": "g", "g0": "g0", "wallflux": "wallflux", "q": "q", "pr": "pr", "drhodtp": "drhodtp", "divu": "divu",
       "rho_stg": "rho_stg", "mu_stg": "mu_stg", "explt0": "explt0", "drhoi_stg": "drhoi_stg"}


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-300))


def _pair(dims, kw):
    from chapsim1ww_amd.heated import HeatedChannel
    from chapsim1ww_amd.solver import ChannelSolver
    sc = props.scale_table(props.synthetic_table())
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    st, tab, n = O.io_case(og, sc, seed=sum(dims))
    s, pt = ChannelSolver(g), props.PropertyTable(sc)
    hc = HeatedChannel(s, pt, **kw)
    hc.upload({MAP[k]: v for k, v in st.items()})
    return st, s, pt, hc, O.OracleIO(og, st, **kw)


@pytest.mark.parametrize("mode", ["auto", "rowtile"])   # x lines through LDS, from global memory
@pytest.mark.parametrize("dims,nflow", [((16, 8, 12), 1), ((36, 9, 20), 3), ((20, 17, 36), 1), ((40, 66, 8), 1),
                                        ((288, 10, 16), 1), ((12, 9, 512), 3), ((16, 300, 8), 1)])
def test_rk_cn_line_lengths(dims, nflow, mode):
    print(f"rk-cn lines {dims} nflow={nflow} {mode}", flush=True)
    st, s, pt, hc, io = _pair(dims, dict(thermal=1, nflow=nflow, visimplicit=1))
    s.set_cn_solver(mode)
    for ns in (1, 2):
        io.prepare(ns)
        io.substep(ns, 1e-3)
        hc.io_prepare(ns)
        hc.solverrk3_mom_io(ns, 1e-3)
        got = hc.download()
        for k in ("g", "g0"):
            assert _rel(got[k], st[k]) < 1e-12, (ns, k, _rel(got[k], st[k]))
    pt.close()
    s.close()


def test_rk_cn_refuses_undivided_cyclic_lines():
    from chapsim1ww_amd.native import CHS_E_ARG, ChsError
    print("rk-cn z lines of 18 rows", flush=True)
    st, s, pt, hc, io = _pair((16, 12, 18), dict(thermal=1, visimplicit=1))
    hc.io_prepare(1)
    with pytest.raises(ChsError) as ei:
        hc.solverrk3_mom_io(1, 1e-3)
    assert ei.value.code == CHS_E_ARG
    pt.close()
    s.close()


@pytest.mark.parametrize("n,nlines", [(48, 32768), (192, 32800), (336, 32769), (384, 32768)])
def test_cyclic_whole_grid_lines(n, nlines):
    """12-row segments of a whole grid's cyclic lines: 32 and 16 lines per
    block, a last block partly filled; the residual of the solution to a few
    eps of |A| |x|."""
    from chapsim1ww_amd.solver import tdma_batched
    print(f"cyclic {n} x {nlines}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(n)
    a, c, r = (torch.rand((n, nlines), dtype=torch.float64, device="cuda", generator=g) - 0.5 for _ in range(3))
    b = 1.0 + a.abs() + c.abs()
    x = r.clone()
    tdma_batched(a, b, c, x, None, n, nlines, nlines, 1, True)
    res = a * x.roll(1, 0) + b * x + c * x.roll(-1, 0) - r
    bound = 64 * 2.0 ** -53 * (a.abs() * x.roll(1, 0).abs() + b * x.abs() + c.abs() * x.roll(-1, 0).abs()).max()
    assert float(res.abs().max()) < float(bound)


def test_tg_thomas_longest_x():
    """The Thomas form's x solve on its longest lines (64 segments, 80 KiB of
    LDS): the substep within 1e-12 of the oracle."""
    from chapsim1ww_amd import fields
    from chapsim1ww_amd.solver import ChannelSolver
    dims = (512, 8, 8)
    print(f"tg thomas {dims}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    st = O.OracleState(og, q, pr, c0)
    dt = 0.4 / st.cfl()
    s = ChannelSolver(g)
    s.set_cn_solver("thomas")
    s.upload_state(q, pr, c0)
    st.substep(1, dt)
    s.solverrk3_mom_tg(1, dt)
    qg, _, cg = s.download_state()
    assert _rel(qg, st.q) < 1e-12 and _rel(cg, st.convh0) < 1e-12, (_rel(qg, st.q), _rel(cg, st.convh0))
    s.close()
