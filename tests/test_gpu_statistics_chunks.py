"""The xz means where their split into chunks of z rows turns: rows of one
chunk (the blocks scale their own sums), of two and of many, x lines below one
wave's 64 lanes, against the NumPy evaluations and tolerances of the statistics
tests."""
import pytest

import test_gpu_statistics as stats

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# L N: below, at and above one and two chunks of 1024 cells; up to 50 chunks
DIMS = [(4, 7, 4), (16, 40, 200), (30, 5, 32), (32, 6, 32), (32, 5, 64), (36, 9, 60), (40, 4, 50), (48, 11, 48),
        (64, 5, 16), (512, 4, 200)]


@pytest.mark.parametrize("dims", DIMS)
def test_tg_chunks(dims):
    stats.test_tg_means_and_maxima(dims)


@pytest.mark.parametrize("dims", DIMS)
def test_io_chunks(dims):
    stats.test_io_means(dims, 1)
