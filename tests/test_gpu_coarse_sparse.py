"""Coarse deposit of few particles a cell, whose rows are staged one behind the
other where a phase of a block holds at most 128: from no particle to twice
that per phase, so that blocks of both stagings lie side by side, in tiles that
are no multiple of the 4-cell block or smaller than it, and with two-byte
positions whose real(4) coordinate rounds (nt >= 128).  Bit for bit against the
oracle."""
import numpy as np
import pytest

from tests.test_gpu_coarse_deposit import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_cell", [0.1, 1.0, 1.8, 3.0])
@pytest.mark.parametrize("nc,nnt,ncb,ix", [(18, 2, 6, 1), (20, 4, 5, 2), (12, 4, 3, 2), (24, 1, 6, 1), (24, 3, 6, 2)])
def test_few_particles(nc, nnt, ncb, ix, per_cell, monkeypatch):
    rng = np.random.default_rng(11)
    n = int(per_cell * nc ** 3)
    pos = rng.random((n, 3)) * nc
    pos[: n // 10] = np.array([nc / nnt, 0.1, nc - 0.2]) + 1.5 * rng.standard_normal((n // 10, 3))
    _check(nc, nnt, ncb, ix, np.mod(pos, nc), None, monkeypatch)


@pytest.mark.parametrize("n", [1, 64, 65, 128, 129, 200])
def test_one_row_full_and_one_more(n, monkeypatch):
    """All of a phase's particles in one or two rows, about the staged batches."""
    rng = np.random.default_rng(n)
    pos = np.array([9.0, 9.0, 9.0]) + rng.random((n, 3)) * np.array([2.0, 1.0, 1.0])
    pos = np.concatenate([pos, np.array([[8.2, 10.3, 9.6], [11.9, 8.8, 9.1]])])
    _check(24, 2, 6, 2, pos, None, monkeypatch)


def test_coordinate_that_rounds(monkeypatch):
    nc = 144
    rng = np.random.default_rng(6)
    cells = np.stack(np.meshgrid(*[np.arange(nc - 24, nc)] * 3, indexing="ij"), -1).reshape(-1, 3)
    c = np.concatenate([cells, rng.integers(0, nc, size=(2000, 3))])
    tops = np.array([0, 32767, 32768, 65535])
    u = np.where(rng.random(c.shape) < 0.7, tops[rng.integers(0, 4, c.shape)], rng.integers(0, 65536, c.shape))
    tempx = (c + (u + 0.5) / 65536.0 - 0.5).astype(np.float32)
    assert ((np.floor(tempx) == c) != (u >= 32768)).sum() > 500
    _check(nc, 1, 6, 2, c + (u + 0.5) / 65536.0, None, monkeypatch)
