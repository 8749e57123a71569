"""xz means and the divergence / CFL maxima on grids that no block or chunk
divides, against vectorised NumPy evaluations of their definitions on the same
fields.  Tolerances: the sums group differently only, 1e-13 of a column's
largest value for the means (sqrt of up to 1e5 terms at 1e-16), equality up to
contraction (1e-14) for the maxima."""
import numpy as np
import pytest

from chapsim1ww_amd import props
from chapsim1ww_amd.grid import ChannelGrid

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

DIMS = [(8, 5, 4), (64, 4, 6), (72, 31, 20), (200, 9, 50), (256, 17, 36), (320, 70, 12), (16, 300, 10)]


def _close(a, b, tol):
    sc = np.abs(b).max(axis=0)
    sc[sc == 0.0] = 1.0
    assert (np.abs(a - b) / sc).max() < tol, (np.abs(a - b) / sc).max()


def _centred(q):
    u, v, w = (q[..., c] for c in range(3))
    return (0.5 * (u + np.roll(u, -1, 0))[:, 1:-1], 0.5 * (v[:, 1:-1] + v[:, 2:]),
            0.5 * (w + np.roll(w, -1, 2))[:, 1:-1])


@pytest.mark.parametrize("dims", DIMS)
def test_tg_means_and_maxima(dims):
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"tg statistics {dims}", flush=True)
    g = ChannelGrid(*dims)
    rng = np.random.default_rng(sum(dims))
    q, pr = np.asfortranarray(rng.standard_normal(g.shape_q)), np.asfortranarray(rng.standard_normal(g.shape_ghost))
    s = ChannelSolver(g)
    s.upload_state(q, pr, None)
    U, P = _centred(q), pr[:, 1:-1]
    cols = [*U, P] + [U[a] * U[b] for a in range(3) for b in range(a, 3)] + [u * P for u in U]
    _close(s.mean_xz(), np.stack([c.mean(axis=(0, 2)) for c in cols], axis=1), 1e-13)
    dy = np.asarray(g.dyfi)[None, :, None]
    u, v, w = (q[..., c] for c in range(3))
    d = ((np.roll(u, -1, 0) - u)[:, 1:-1] * g.dxi, (v[:, 2:] - v[:, 1:-1]) * dy, (np.roll(w, -1, 2) - w)[:, 1:-1] * g.dzi)
    assert abs(s.divgck() / np.abs(d[0] + d[1] + d[2]).max() - 1.0) < 1e-14
    cfl = np.abs(U[0] * g.dxi) + np.abs(U[1] * dy) + np.abs(U[2] * g.dzi)
    assert abs(s.cfl() / cfl.max() - 1.0) < 1e-14
    q[dims[0] - 1, dims[1], dims[2] - 1, 2] = np.nan   # the last cell: both maxima propagate it
    s.upload_state(q, None, None)
    assert np.isnan(s.divgck()) and np.isnan(s.cfl())
    s.close()


@pytest.mark.parametrize("dims", DIMS)
@pytest.mark.parametrize("thermal", [0, 1])
def test_io_means(dims, thermal):
    from chapsim1ww_amd.heated import HeatedChannel
    from chapsim1ww_amd.solver import ChannelSolver
    print(f"io statistics {dims} thermal={thermal}", flush=True)
    g = ChannelGrid(*dims)
    s = ChannelSolver(g)
    pt = props.PropertyTable(props.scale_table(props.synthetic_table(64)))
    hc = HeatedChannel(s, pt, thermal=thermal)
    rng = np.random.default_rng(sum(dims) + 1)
    f = {k: rng.standard_normal(hc.shapes[k]) for k in ("q", "g", "pr", "temperature", "density", "enthalpy",
                                                        "viscosity")}
    hc.upload(f)
    U, G, P = _centred(f["q"]), _centred(f["g"]), f["pr"][:, 1:-1]
    T, D, H, V = (f[k][:, 1:-1] for k in ("temperature", "density", "enthalpy", "viscosity"))
    pairs = [(a, b) for a in range(3) for b in range(a, 3)]
    cols = [*U, P, *G] + [u * P for u in U] + [U[a] * U[b] for a, b in pairs] + [U[a] * G[b] for a, b in pairs]
    th = [T, D, H, V, T * T, D * D, H * H, H * D, H * P] + [H * u for u in U] + [H * q for q in G]
    cols += th if thermal else [np.zeros_like(c) for c in th]
    _close(hc.mean_xz_io(), np.stack([c.mean(axis=(0, 2)) for c in cols], axis=1), 1e-13)
    pt.close()
    s.close()
