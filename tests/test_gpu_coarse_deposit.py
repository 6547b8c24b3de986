"""Coarse deposit at the edges of its blocks: tiles that are no multiple of the
4-cell block, tiles smaller than one, and two-byte positions in a tile wide
enough that the reference's real(4) coordinate rounds (nt >= 128), where codes
just below a half-cell round onto it; each staged (default), with every phase
term by term (CUBE_CD_HEAVY=0) and mixed.  Bit for bit against the oracle."""
import numpy as np
import pytest

from cafproject_amd import ics
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _check(nc, nnt, ncb, ix, pos, heavy, monkeypatch):
    from cafproject_amd.cube import Cube
    if heavy is not None:
        monkeypatch.setenv("CUBE_CD_HEAVY", heavy)
    st = ics.disjoint_state(pos, np.zeros_like(pos, dtype=np.float32), nc, nnt, izipx=ix, izipv=2, sigma_vi=1.0)
    np_nc = max(2, int(np.ceil((len(pos) / nc ** 3) ** (1 / 3))))
    oc = O.OracleCube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=2, tile_buffer=30.0, image_buffer=30.0)
    oc.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    oc.buffer_grid(); oc.buffer_x(); oc.buffer_v()
    g = Cube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=2)
    g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    m = 0.75
    t = g.coarse_deposit(m)
    r3, s = oc.coarse_deposit(m)
    assert np.array_equal(g.get_field("rho_c"), r3)
    assert abs(t / s - 1) < 1e-12


@pytest.mark.parametrize("heavy", [None, "0", "300"])
@pytest.mark.parametrize("nc,nnt,ncb,ix", [(18, 2, 6, 1), (20, 4, 5, 2), (16, 4, 4, 1), (12, 4, 3, 2), (20, 1, 6, 1)])
def test_tiles_and_blocks(nc, nnt, ncb, ix, heavy, monkeypatch):
    rng = np.random.default_rng(7)
    n = 8 * nc ** 3
    pos = rng.random((n, 3)) * nc
    # a halo across a tile corner and one inside a block; empty cells besides
    pos[: n // 5] = np.array([nc / nnt, 0.1, nc - 0.2]) + 0.4 * rng.standard_normal((n // 5, 3))
    pos[n // 5: n // 4] = np.array([2.5, 2.5, 3.0]) + 0.1 * rng.standard_normal((n // 4 - n // 5, 3))
    _check(nc, nnt, ncb, ix, np.mod(pos, nc), heavy, monkeypatch)


@pytest.mark.parametrize("heavy", [None, "0"])
def test_coordinate_that_rounds(heavy, monkeypatch):
    nc = 144
    rng = np.random.default_rng(5)
    cells = np.stack(np.meshgrid(*[np.arange(nc - 20, nc)] * 3, indexing="ij"), -1).reshape(-1, 3)
    c = np.repeat(np.concatenate([cells, rng.integers(0, nc, size=(500, 3))]), 3, axis=0)
    tops = np.array([0, 32767, 32768, 65535])
    u = np.where(rng.random(c.shape) < 0.7, tops[rng.integers(0, 4, c.shape)], rng.integers(0, 65536, c.shape))
    # the premise: the rounded coordinate of some particles is in another half than their code
    tempx = (c + (u + 0.5) / 65536.0 - 0.5).astype(np.float32)
    assert ((np.floor(tempx) == c) != (u >= 32768)).sum() > 1000
    _check(nc, 1, 6, 2, c + (u + 0.5) / 65536.0, heavy, monkeypatch)
