"""Batched line solves at the sizes where the choice of kernel turns: short
cyclic lines of whole segments (the serial sweep of their reduced systems, 4, 8
and 12 rows a segment, both lane orders), the line counts at which the blocks
grow, pitches that straddle the 128-byte lines, and padded layouts in which
neither the lines nor the rows are adjacent, against the CPU oracle.  Tolerance:
the FP64 parity bound of the other line tests (1e-12 of the largest value) for
systems with |a| + |c| < b; entries between the lines stay as they are."""
import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _check(n, nl, es, ls, cyclic, seed):
    from chapsim1ww_amd import solver
    rng = np.random.default_rng(seed)
    size = (n - 1) * es + (nl - 1) * ls + 1
    a, c = rng.uniform(-0.9, -0.1, size), rng.uniform(-0.9, -0.1, size)
    b, d = 2.0 + np.abs(rng.standard_normal(size)), rng.standard_normal(size)
    bc = None if cyclic else np.asfortranarray(rng.standard_normal((nl, 2)))
    ref = d.copy()
    if cyclic:
        O.tdma_cyc(a, b, c, ref, n, nl, es, ls)
    else:
        O.tdma_noncyc(a, b, c, ref, bc, n, nl, es, ls)
    dev = [None if v is None else torch.from_numpy(v.ravel(order="F").copy()).cuda() for v in (a, b, c, d, bc)]
    solver.tdma_batched(*dev, n, nl, es, ls, cyclic)
    out = dev[3].cpu().numpy()
    assert np.abs(out - ref).max() < 1e-12 * np.abs(ref).max()
    used = np.zeros(size, bool)
    used[(np.arange(nl)[:, None] * ls + np.arange(n)[None, :] * es).ravel()] = True
    assert np.array_equal(out[~used], d[~used])


@pytest.mark.parametrize("n", [4, 8, 12, 16, 20, 24, 28, 32, 40, 56, 64, 72, 80, 88, 96, 104, 128, 132, 192, 288, 320,
                               384])
@pytest.mark.parametrize("nl", [37, 1279, 4096, 4099, 8208, 8209])
@pytest.mark.parametrize("march", ["IJJ", "IJI"])
def test_cyclic_plans(n, nl, march):
    print(f"cyclic n={n} nlines={nl} {march}", flush=True)
    es, ls = (nl, 1) if march == "IJJ" else (1, n)
    _check(n, nl, es, ls, True, 7 * n + nl)


@pytest.mark.parametrize("n,nl", [(17, 14000), (37, 14003), (125, 14001), (128, 14000), (8, 40000), (12, 14001), (20, 14000), (28, 14000), (24, 8193), (64, 32800),
                                  (96, 16400), (80, 16385), (128, 16399), (192, 40000)])
@pytest.mark.parametrize("march", ["IJJ", "IJI"])
@pytest.mark.parametrize("cyclic", [True, False])
def test_many_lines(n, nl, march, cyclic):
    print(f"many n={n} nlines={nl} {march} cyclic={cyclic}", flush=True)
    es, ls = (nl, 1) if march == "IJJ" else (1, n)
    _check(n, nl, es, ls, cyclic, n + nl)


@pytest.mark.parametrize("n", [9, 16, 17, 32, 33, 64, 65, 96, 128, 129, 192, 256, 257, 360, 385])
@pytest.mark.parametrize("nl", [1279, 1280, 4097, 8208, 8209])
def test_noncyclic_plans(n, nl):
    print(f"non-cyclic n={n} nlines={nl}", flush=True)
    _check(n, nl, nl, 1, False, 3 * n + nl)


@pytest.mark.parametrize("cyclic", [True, False])
@pytest.mark.parametrize("n,nl,es,ls", [(24, 5000, 5008, 1), (24, 9000, 9003, 1), (40, 300, 1, 43), (24, 130, 2, 51),
                                        (12, 70, 3, 37), (96, 4100, 3, 290), (17, 33, 70, 2)])
def test_padded_layouts(n, nl, es, ls, cyclic):
    print(f"padded n={n} nlines={nl} es={es} ls={ls} cyclic={cyclic}", flush=True)
    _check(n, nl, es, ls, cyclic, n + nl + es)
