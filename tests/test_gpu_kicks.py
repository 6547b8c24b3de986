"""A step's two kicks in one pass over 4x2x2 blocks of coarse cells, against the
stages one by one (a fine kick, then a coarse one, gathering from global
memory): tiles that are no multiple of the block or smaller than it, crowded
and empty cells, and two-byte positions in a tile wide enough (nt > 128) that
the reference's real(4) coordinate rounds onto the next cell.  Bit for bit."""
import numpy as np
import pytest

from cafproject_amd import ics

pytestmark = pytest.mark.gpu


def _state(nc, nnt, ix, iv, pos, rng):
    v = (0.02 * rng.standard_normal(pos.shape)).astype(np.float32)
    return ics.disjoint_state(pos, v, nc, nnt, izipx=ix, izipv=iv)


def _check(nc, nnt, ncb, ix, iv, pos, rng):
    from cafproject_amd.cube import Cube
    st = _state(nc, nnt, ix, iv, pos, rng)
    np_nc = max(2, int(np.ceil((len(pos) / nc ** 3) ** (1 / 3))))
    m, s0 = 0.75, st["sigma_vi"]
    s1, a_mid, dt = float(np.float32(1.02 * s0)), 0.1, 4.0
    out = []
    for one in (True, False):
        g = Cube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=iv)
        g.init_kernels()
        g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
        if one:
            vmax = g.particle_mesh(a_mid, dt, s0, s1, m)["vmax"]
        else:
            g.fine_deposit(m)
            g.fine_force()
            g.fine_kick(a_mid, dt, s0, s1)
            g.coarse_deposit(m)
            g.coarse_force()
            vmax = g.coarse_kick(a_mid, dt, s1)
        out.append((g.get_state()["vp"], np.array(vmax, np.float32)))
        del g
    assert not np.array_equal(out[0][0], st["vp"])
    assert np.array_equal(out[0][0], out[1][0])
    assert np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("ix,iv", [(1, 2), (2, 1)])
@pytest.mark.parametrize("nc,nnt,ncb", [(18, 2, 6), (20, 4, 5), (12, 4, 3), (20, 1, 6)])
def test_tiles_and_blocks(nc, nnt, ncb, ix, iv):
    rng = np.random.default_rng(13)
    n = 8 * nc ** 3
    pos = rng.random((n, 3)) * nc
    pos[: n // 5] = np.array([nc / nnt, 0.1, nc - 0.2]) + 0.4 * rng.standard_normal((n // 5, 3))
    _check(nc, nnt, ncb, ix, iv, np.mod(pos, nc), rng)


def test_coordinate_that_rounds():
    nc = 144
    rng = np.random.default_rng(5)
    cells = np.stack(np.meshgrid(*[np.arange(nc - 20, nc)] * 3, indexing="ij"), -1).reshape(-1, 3)
    c = np.repeat(np.concatenate([cells, rng.integers(0, nc, size=(500, 3))]), 3, axis=0)
    tops = np.array([0, 16383, 16384, 49152, 65535])
    u = np.where(rng.random(c.shape) < 0.7, tops[rng.integers(0, len(tops), c.shape)], rng.integers(0, 65536, c.shape))
    # the premise: the rounded coordinate of some particles is past their cell
    tempx = (4 * c + (u + 0.5) / 16384.0).astype(np.float32)
    assert (np.floor(tempx) == 4 * c + 4).sum() > 1000
    _check(nc, 1, 6, 2, 2, c + (u + 0.5) / 65536.0, rng)
