"""Fine deposit at the edges of its blocks: tiles that are no multiple of the
4-cell block, tiles smaller than one, and two-byte positions in a tile wide
enough that the reference's real(4) coordinate rounds (nt > 128), where the top
code of a fine sub-cell rounds onto the next; with crowded cells on their own
(default), every cell so (CUBE_FD_HEAVY=0) and none, where a crowded block's
rows take several rounds of staging.  Bit for bit against the oracle."""
import numpy as np
import pytest

from cafproject_amd import ics
from oracle import oracle as O

pytestmark = pytest.mark.gpu
HEAVY = [None, "0", "1000000000"]


def _check(nc, nnt, ncb, ix, pos, heavy, monkeypatch):
    from cafproject_amd.cube import Cube
    if heavy is not None:
        monkeypatch.setenv("CUBE_FD_HEAVY", heavy)
    st = ics.disjoint_state(pos, np.zeros_like(pos, dtype=np.float32), nc, nnt, izipx=ix, izipv=2, sigma_vi=1.0)
    np_nc = max(2, int(np.ceil((len(pos) / nc ** 3) ** (1 / 3))))
    oc = O.OracleCube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=2, tile_buffer=30.0, image_buffer=30.0)
    oc.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    oc.buffer_grid(); oc.buffer_x(); oc.buffer_v()
    g = Cube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=2)
    g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    m = 0.75
    s, nfb, nft = 0.0, oc.nfb, oc.nft
    rf = np.empty((4 * nc,) * 3, np.float32)  # the tiles' interiors, side by side
    for tz in range(nnt):
        for ty in range(nnt):
            for tx in range(nnt):
                rho, part = oc.fine_deposit(tx + 1, ty + 1, tz + 1, m)
                s += part
                rf[tz * nft:(tz + 1) * nft, ty * nft:(ty + 1) * nft, tx * nft:(tx + 1) * nft] = \
                    rho[nfb:nfb + nft, nfb:nfb + nft, nfb:nfb + nft]
    for _ in range(2):  # the list of crowded cells is empty again
        t = g.fine_deposit(m)
        assert np.array_equal(g.get_field("rho_f"), rf)
        # two sums of nf^3 terms >= 0, each off by at most nf^3 roundings
        assert abs(t / s - 1) < 2 * (4 * nc) ** 3 * 2.0 ** -53


@pytest.mark.parametrize("heavy", HEAVY)
@pytest.mark.parametrize("nc,nnt,ncb,ix", [(18, 2, 6, 1), (20, 4, 5, 2), (16, 4, 4, 1), (12, 4, 3, 2), (20, 1, 6, 1)])
def test_tiles_and_blocks(nc, nnt, ncb, ix, heavy, monkeypatch):
    rng = np.random.default_rng(11)
    n = 8 * nc ** 3
    pos = rng.random((n, 3)) * nc
    # a halo across a tile corner and one inside a block; empty cells besides
    pos[: n // 5] = np.array([nc / nnt, 0.1, nc - 0.2]) + 0.4 * rng.standard_normal((n // 5, 3))
    pos[n // 5: n // 4] = np.array([2.5, 2.5, 3.0]) + 0.1 * rng.standard_normal((n // 4 - n // 5, 3))
    _check(nc, nnt, ncb, ix, np.mod(pos, nc), heavy, monkeypatch)


@pytest.mark.parametrize("heavy", HEAVY)
def test_coordinate_that_rounds(heavy, monkeypatch):
    nc = 144
    rng = np.random.default_rng(5)
    cells = np.stack(np.meshgrid(*[np.arange(nc - 20, nc)] * 3, indexing="ij"), -1).reshape(-1, 3)
    c = np.repeat(np.concatenate([cells, rng.integers(0, nc, size=(500, 3))]), 3, axis=0)
    tops = np.array([0, 16383, 16384, 32767, 49151, 49152, 65535])
    u = np.where(rng.random(c.shape) < 0.7, tops[rng.integers(0, len(tops), c.shape)], rng.integers(0, 65536, c.shape))
    # the premise: the rounded coordinate of some particles is in another sub-cell than their code
    tempx = (4 * c + (u + 0.5) / 16384.0).astype(np.float32)
    assert ((np.floor(tempx) - 4 * c) != (u >> 14)).sum() > 1000
    _check(nc, 1, 6, 2, c + (u + 0.5) / 65536.0, heavy, monkeypatch)
