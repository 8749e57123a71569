"""FP64 Poisson solves over the FFT lengths of the register transforms: every
radix of both stages (2..16), three-stage lengths, blocks of several rows j
with a remainder, row pairs that do not fill the last block, and lengths
without a register plan, against the CPU oracle.  Tolerance: the FP64 parity
bound of the other Poisson tests, 1e-12 of the largest value."""
import numpy as np
import pytest

import oracle as O
from chapsim1ww_amd import fields
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 5, 6), (6, 7, 4), (8, 5, 10), (10, 9, 8), (12, 4, 18), (18, 6, 12), (20, 5, 30),
                                  (24, 11, 16), (30, 5, 24), (32, 6, 20), (36, 7, 40), (40, 5, 36), (48, 9, 32),
                                  (50, 5, 54), (54, 6, 50), (60, 5, 48), (64, 13, 60), (72, 5, 64), (80, 6, 90),
                                  (90, 5, 72), (96, 5, 100), (100, 6, 80), (108, 5, 96), (120, 7, 128), (128, 5, 120),
                                  (144, 5, 150), (150, 6, 144), (160, 5, 180), (180, 5, 160), (192, 6, 240),
                                  (240, 5, 192), (200, 5, 250), (250, 5, 200), (216, 5, 270), (288, 5, 320),
                                  (320, 5, 288), (360, 4, 384), (384, 5, 360), (400, 4, 432), (432, 4, 400),
                                  (450, 4, 480), (480, 5, 486), (512, 4, 500), (500, 4, 512), (600, 4, 540),
                                  (648, 4, 16), (256, 5, 96), (96, 5, 256)])
def test_poisson_fp64_lengths(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"poisson fp64 {dims}", flush=True)
    g, og = ChannelGrid(*dims), O.OracleGrid(*dims)
    f = fields.poisson_rhs(g, seed=sum(dims))
    ref = O.poisson(og, f)
    s = ChannelSolver(g, "fp64")
    df = torch.from_numpy(np.asfortranarray(f).ravel(order="F").copy()).cuda()
    dph = torch.full((g.L * (g.M + 2) * g.N,), 7.0, dtype=torch.float64, device="cuda")
    s.fft99_pois3d(df, dph)
    out = dph.cpu().numpy().reshape(g.shape_ghost, order="F")
    assert np.abs(out - ref).max() < 1e-12 * np.abs(ref).max()
    assert np.all(out[:, 0, :] == 0.0) and np.all(out[:, -1, :] == 0.0)
    s.close()
