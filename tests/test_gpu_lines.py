"""Batched line solves at the edges of their configurations: cyclic lines of
any length (the split-off last unknown), lines long enough for the smallest
blocks and the one-thread-per-line form behind them, few and many lines, both
layouts, against the CPU oracle.  Tolerance: the FP64 parity bound of the
other line tests (1e-12 of the largest value) for systems with |a| + |c| < b."""
import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cyclic", [True, False])
@pytest.mark.parametrize("march", ["IJJ", "IJI"])
@pytest.mark.parametrize("n,nl", [(3, 70), (8, 9), (9, 33), (10, 2050), (17, 5), (135, 1500), (191, 2048), (250, 3),
                                  (255, 40000), (252, 32768), (257, 64), (511, 130), (513, 67), (1024, 40),
                                  (1025, 21), (2047, 9), (2048, 5), (2049, 6), (2050, 4)])
def test_line_lengths(n, nl, march, cyclic):
    from chapsim1ww_amd import solver
    print(f"lines n={n} nlines={nl} {march} cyclic={cyclic}", flush=True)
    rng = np.random.default_rng(31 * n + nl)
    shape, es, ls = ((nl, n), nl, 1) if march == "IJJ" else ((n, nl), 1, n)
    a = np.asfortranarray(rng.uniform(-0.9, -0.1, shape))
    c = np.asfortranarray(rng.uniform(-0.9, -0.1, shape))
    b = np.asfortranarray(2.0 + np.abs(rng.standard_normal(shape)))
    d = np.asfortranarray(rng.standard_normal(shape))
    bc = None if cyclic else np.asfortranarray(rng.standard_normal((nl, 2)))
    ref = d.copy(order="F")
    if cyclic:
        O.tdma_cyc(a, b, c, ref, n, nl, es, ls)
    else:
        O.tdma_noncyc(a, b, c, ref, bc, n, nl, es, ls)
    dev = [None if v is None else torch.from_numpy(v.ravel(order="F").copy()).cuda() for v in (a, b, c, d, bc)]
    solver.tdma_batched(*dev, n, nl, es, ls, cyclic)
    out = dev[3].cpu().numpy().reshape(shape, order="F")
    assert np.abs(out - ref).max() < 1e-12 * np.abs(ref).max()
