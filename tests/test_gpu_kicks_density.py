"""A step's two kicks in one pass on either side of the density where they turn
from gathering row by row to blocks with the mesh in LDS, against the oracle's
kicks on the same force meshes, and in blocks of a tile of 144 cells with
two-byte positions, whose real(4) coordinates round.  Bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_kicks_oracle import _check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ix,iv", [(1, 1), (2, 2)])
@pytest.mark.parametrize("nc,nnt,ncb", [(32, 2, 6), (48, 3, 6), (24, 1, 6)])
@pytest.mark.parametrize("per_cell", [0.2, 1.0, 2.49, 2.51])
def test_densities(nc, nnt, ncb, ix, iv, per_cell):
    rng = np.random.default_rng(29)
    n = int(per_cell * nc ** 3)
    pos = rng.random((n, 3)) * nc
    pos[: n // 5] = np.array([nc / nnt, 0.1, nc - 0.2]) + 0.4 * rng.standard_normal((n // 5, 3))
    _check(nc, nnt, ncb, ix, iv, np.mod(pos, nc), rng)


def test_blocks_of_a_wide_tile():
    nc = 144
    rng = np.random.default_rng(6)
    n = int(2.52 * nc ** 3)
    c = rng.integers(0, nc, size=(n, 3))
    tops = np.array([0, 16383, 16384, 49152, 65535])
    u = rng.integers(0, 65536, size=(n, 3))
    u[: n // 4] = tops[rng.integers(0, len(tops), (n // 4, 3))]
    _check(nc, 1, 6, 2, 2, c + (u + 0.5) / 65536.0, rng)
