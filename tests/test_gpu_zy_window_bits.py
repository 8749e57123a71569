"""The z and y window solves of the mixed form in one pass and in two: the same
expressions in the same order, so the same state to the last bit, with window
widths 4 and 8 in z and 4, 8 and 12 in y, tiles that the grid does not fill, and
mass flux along x and z (the correction subtracted on load)."""
import numpy as np
import pytest

from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,fac,nflow", [((48, 20, 64), 0.4, 1), ((64, 40, 128), 0.4, 3), ((80, 33, 64), 0.1, 1),
                                            ((240, 66, 64), 0.4, 1), ((96, 130, 128), 0.8, 1)])
def test_mixed_windows_bit_for_bit(dims, fac, nflow):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"zy window bits {dims} {fac} {nflow}", flush=True)
    g = ChannelGrid(*dims)
    q, pr, c0 = fields.init_tg_fields(g, seed=3)
    out = []
    for mode in ("auto", "marching"):
        s = ChannelSolver(g, "mixed", nflow=nflow)
        s.set_cn_solver(mode)
        s.upload_state(q, pr, c0)
        dt = fac / s.cfl()
        info = s.cn_info(1, dt)
        assert info["path"] == "stencil" and info["kz"] <= 8 and info["ky"] <= 12, info
        s.solverrk3_mom_tg(0, dt)
        s.solverrk3_mom_tg(1, dt)
        out.append((*s.download_state(), info))
        s.close()
    print(out[0][3], flush=True)
    for a, b in zip(out[0][:3], out[1][:3]):
        assert np.array_equal(a, b)
