"""Property records loaded by quads and pairs of lanes and the T interval taken
from H's: calls around the lines between the lookup's forms and rows whose
ends leave parts of quads, with neighbouring cells far apart in the table, on
knots, outside the table and NaN.  Outputs equal the CPU oracle bit for bit."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import native as nat
from chapsim1ww_amd import props

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [2, 3, 1027, (1 << 20) - 1, (1 << 20) + 1, (3 << 21) - 3, (3 << 21) + 8191])
@pytest.mark.parametrize("with_cp", [True, False])
def test_quads_bitwise(cells, with_cp):
    print(f"quads cells={cells} cp={with_cp}", flush=True)
    knots = 2048
    sc = props.scale_table(props.synthetic_table(knots))
    rng = np.random.default_rng(cells)
    H = np.asarray(sc["H"])
    h = rng.uniform(H[0] + 1e-9, H[-1] - 1e-9, cells)
    k = rng.random(cells)
    on = k < 0.2   # knots and their neighbours: T rounds past a knot
    h[on] = H[rng.integers(1, knots - 1, on.sum())]
    up = k < 0.1
    h[up] = np.nextafter(h[up], np.inf)
    if cells > 1000:
        h[(k > 0.9) & (k < 0.92)] = np.nan
        h[k > 0.98] = 0.0   # left as they are
    tab, n = O.build_prop_tab(sc), knots
    if isinstance(tab, tuple):
        tab, n = tab
    ref = [np.full(cells, 3.0) for _ in range(5)]
    O.therm_prop_update(tab, n, h, *ref[:4], ref[4] if with_cp else None)
    pt = props.PropertyTable(sc)
    out = [torch.full((cells,), 3.0, dtype=torch.float64, device="cuda") for _ in range(5)]
    hd = torch.from_numpy(h).cuda()
    assert pt.update(hd, *out[:4], out[4] if with_cp else None) == 0
    for a, b in zip(out, ref):
        assert np.array_equal(a.cpu().numpy(), b, equal_nan=True)
    if cells > 1000:   # some cells of a quad outside the table: the others are still right
        bad = torch.arange(5, 900, 3)
        hd[bad] = float(H[-1]) + 1.0
        ok = torch.ones(cells, dtype=torch.bool)
        ok[bad] = False
        out2 = [torch.full_like(o, 3.0) for o in out]
        with pytest.raises(nat.ChsError, match=f"{len(bad)} cells outside"):
            pt.update(hd, *out2[:4], out2[4] if with_cp else None)
        for a, b in zip(out2, ref):
            assert np.array_equal(a.cpu().numpy()[ok.numpy()], b[ok.numpy()], equal_nan=True)
            assert (a.cpu()[bad] == 3.0).all()
    pt.close()
