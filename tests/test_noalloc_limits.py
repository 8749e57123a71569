"""chs_tdma_batched_noalloc's limit on the lines its header names, refused on the
host: cyclic lengths no segments divide, four-row ones beyond 128 rows,
non-cyclic lines of more than 512 rows, all one line above 4194304 / (3 n).  The
kernels of these lines need no workspace, and the message does not say so."""
import pytest

from chapsim1ww_amd import native as nat

LIMIT = 4194304


@pytest.mark.parametrize("n,cyclic", [(7, 1), (135, 1), (140, 1), (260, 1), (388, 1), (513, 0), (600, 0),
                                      (2100, 0), (2100, 1)])
def test_refused_above_the_limit(n, cyclic):
    lib = nat.load()
    nl = LIMIT // (3 * n) + 1
    rc = lib.chs_tdma_batched_noalloc(1, 1, 1, 1, None, n, nl, nl, 1, cyclic, None)
    msg = lib.chs_last_error().decode()
    assert rc == nat.CHS_E_ARG and "held to 3*n*nlines <= 4194304" in msg and "need a workspace" not in msg
