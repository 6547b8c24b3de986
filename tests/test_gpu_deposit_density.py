"""Both deposits over the densities at which their staging changes (rows of few
particles one behind the other, a batch of 64 slots each, or of many one behind
the other in more batches): the same sums on either side of each line, in tiles
that are no multiple of the 4-cell block or smaller than it, with empty cells
and crowded ones, these on their own (default) and with the others; and in a
tile of 144 cells with two-byte positions, whose real(4) coordinates round.
Bit for bit against the oracle."""
import numpy as np
import pytest

from tests.test_gpu_coarse_deposit import _check as coarse
from tests.test_gpu_fine_deposit import _check as fine

pytestmark = pytest.mark.gpu


def _positions(nc, nnt, per_cell, rng):
    n = max(1, int(per_cell * nc ** 3))
    pos = rng.random((n, 3)) * nc
    pos[: n // 10] = np.array([nc / nnt, 0.1, nc - 0.2]) + 1.5 * rng.standard_normal((n // 10, 3))
    pos[n // 10: n // 8] = np.array([2.5, 2.5, 3.0]) + 0.3 * rng.standard_normal((n // 8 - n // 10, 3))
    return np.mod(pos, nc)


@pytest.mark.parametrize("heavy", [None, "1000000000"])
@pytest.mark.parametrize("per_cell", [0.1, 1.0, 2.55, 2.57, 12.7, 12.9, 27.0, 40.0])
@pytest.mark.parametrize("nc,nnt,ncb,ix", [(18, 2, 6, 1), (20, 4, 5, 2), (12, 4, 3, 2), (24, 1, 6, 1)])
def test_fine(nc, nnt, ncb, ix, per_cell, heavy, monkeypatch):
    fine(nc, nnt, ncb, ix, _positions(nc, nnt, per_cell, np.random.default_rng(17)), heavy, monkeypatch)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 128, 256, 257, 1500, 1600])
def test_fine_rows_full_and_one_more(n, monkeypatch):
    """All particles in one row of cells, about the staged batches."""
    rng = np.random.default_rng(n)
    pos = np.array([9.0, 9.0, 9.0]) + rng.random((n, 3)) * np.array([3.0, 1.0, 1.0])
    fine(24, 2, 6, 2, np.concatenate([pos, np.array([[8.2, 10.3, 9.6], [11.9, 8.8, 9.1]])]), "1000000000", monkeypatch)


def test_wide_tile(monkeypatch):
    nc = 144
    rng = np.random.default_rng(8)
    n = int(2.6 * nc ** 3)  # a batch a row in both
    c = rng.integers(0, nc, size=(n, 3))
    tops = np.array([0, 16383, 16384, 32767, 32768, 49151, 49152, 65535])
    u = rng.integers(0, 65536, size=(n, 3))
    u[: n // 4] = tops[rng.integers(0, len(tops), (n // 4, 3))]
    pos = c + (u + 0.5) / 65536.0
    coarse(nc, 1, 6, 2, pos, None, monkeypatch)
    fine(nc, 1, 6, 2, pos, None, monkeypatch)
