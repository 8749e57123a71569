"""THERM_PROP_UPDATE and the energy substep through every form of the property
lookup: small calls (one cell per thread), large ones with the coefficient
records in LDS (tables up to about 2100 knots) and with them in global memory
(larger tables), at sizes around the blocks' chunks.  Outputs equal the CPU
oracle bit for bit, as the lookups evaluate the same expressions."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import native as nat
from chapsim1ww_amd import props

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("knots", [5, 600, 2048, 4096])
@pytest.mark.parametrize("cells", [1, 255, 257, 8193, (3 << 19) - 1, (3 << 19) + 4097])
@pytest.mark.parametrize("with_cp", [True, False])
def test_lookup_forms_bitwise(knots, cells, with_cp):
    print(f"lookup knots={knots} cells={cells} cp={with_cp}", flush=True)
    sc = props.scale_table(props.synthetic_table(knots))
    rng = np.random.default_rng(knots + cells)
    h = rng.uniform(sc["H"][0] + 1e-9, sc["H"][-1] - 1e-9, cells)
    h[0] = np.nan if cells > 300 else h[0]
    if cells > 300:
        h[1], h[2] = 0.0, 5e-11   # left as they are
    tab = O.build_prop_tab(sc)
    tab, n = tab if isinstance(tab, tuple) else (tab, knots)
    ref = [np.full(cells, 3.0) for _ in range(5)]
    O.therm_prop_update(tab, n, h, *ref[:4], ref[4] if with_cp else None)
    pt = props.PropertyTable(sc)
    out = [torch.full((cells,), 3.0, dtype=torch.float64, device="cuda") for _ in range(5)]
    hd = torch.from_numpy(h).cuda()
    for _ in range(2):   # the counters are clear again after a call
        assert pt.update(hd, *out[:4], out[4] if with_cp else None) == 0
    for a, b in zip(out, ref):
        assert np.array_equal(a.cpu().numpy(), b, equal_nan=True)
    hd[cells // 2] = float(sc["H"][-1]) + 1.0
    with pytest.raises(nat.ChsError, match="1 cells outside"):
        pt.update(hd, *out[:4])
    hd[cells // 2] = float(sc["H"][1])
    pt.update(hd, *out[:4])
    pt.close()


@pytest.mark.parametrize("knots", [1000, 3000])
def test_energy_substep_forms_bitwise(knots):
    from chapsim1ww_amd.grid import ChannelGrid
    from chapsim1ww_amd.energy import ThermalState
    from chapsim1ww_amd.solver import ChannelSolver
    dims = (24, 20, 16)
    sc = props.scale_table(props.synthetic_table(knots))
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    st, tab, n = O.thermal_case(og, sc, seed=3)
    s, pt = ChannelSolver(g), props.PropertyTable(sc)
    ts = ThermalState(s, pt)
    names = dict(rhoh="rhoh", enthalpy="h", temperature="T", density="rho", density0="rho0", density1="rho1",
                 viscosity="mu", viscosity0="mu0", thermcondt="kap", rhs_energy0="rhs0", g="g", g0="g0",
                 wallflux="wallflux")
    ts.upload({k: st[v] for k, v in names.items()})
    for ns in (1, 2, 3):
        O.energy_substep(og, st, tab, n, ns, 1e-3, 1.0 / 2800.0, O.rhoh_max(sc))
        ts.solverrk3_eng_io(ns, 1e-3, 1.0 / 2800.0)
        pt.check()
    got = ts.download()
    for k, v in names.items():
        assert np.array_equal(got[k], st[v]), k
    pt.close()
    s.close()
