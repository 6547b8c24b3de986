"""A step's two kicks in one pass over 4x2x2 blocks of coarse cells against the
oracle's kicks on the same force meshes: tiles that are no multiple of the block
or smaller than it, crowded and empty cells, and two-byte positions in a tile
wide enough (nt > 128) that the reference's real(4) coordinate rounds onto the
next cell.  Codes and v_max bit for bit."""
import numpy as np
import pytest

from cafproject_amd import ics
from oracle import oracle as O
from tests.helpers import global_force_to_tile

pytestmark = pytest.mark.gpu


def _check(nc, nnt, ncb, ix, iv, pos, rng):
    from cafproject_amd.cube import Cube
    v = (0.02 * rng.standard_normal(pos.shape)).astype(np.float32)
    st = ics.disjoint_state(pos, v, nc, nnt, izipx=ix, izipv=iv)
    state = (st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    np_nc = max(2, int(np.ceil((len(pos) / nc ** 3) ** (1 / 3))))
    m, s0, a_mid, dt = 0.75, st["sigma_vi"], 0.1, 4.0
    s1 = float(np.float32(1.02 * s0))
    g = Cube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=iv)
    g.init_kernels()
    g.set_state(*state)
    g.fine_deposit(m)
    g.fine_force()
    ff = g.get_field("force_f")
    g.coarse_deposit(m)
    g.coarse_force()
    fc = g.get_field("force_c")
    vmax = g.particle_mesh(a_mid, dt, s0, s1, m)["vmax"]
    oc = O.OracleCube(nc, nnt, ncb=ncb, np_nc=np_nc, izipx=ix, izipv=iv, tile_buffer=30.0, image_buffer=30.0)
    oc.set_state(*state)
    oc.buffer_grid(); oc.buffer_x(); oc.buffer_v()
    for itz in range(1, nnt + 1):
        for ity in range(1, nnt + 1):
            for itx in range(1, nnt + 1):
                tile = global_force_to_tile(ff, nc, nnt, itx, ity, itz)
                O.lib().oc_fine_kick(oc._c, itx, ity, itz, O._p(tile), a_mid, dt, s0, s1)
    halo = np.ascontiguousarray(np.pad(fc, ((1, 1), (1, 1), (1, 1), (0, 0)), mode="wrap"))
    vo = np.zeros(3, np.float32)
    O.lib().oc_coarse_kick(oc._c, O._p(halo), a_mid, dt, s1, O._p(vo))
    got = g.get_state()["vp"]
    assert not np.array_equal(got, st["vp"])
    assert np.array_equal(got, oc.get_state()["vp"])
    assert np.array_equal(np.asarray(vmax, np.float32), vo)


@pytest.mark.parametrize("ix,iv", [(1, 2), (2, 1)])
@pytest.mark.parametrize("nc,nnt,ncb", [(18, 2, 6), (20, 4, 5), (12, 4, 3), (20, 1, 6)])
def test_tiles_and_blocks(nc, nnt, ncb, ix, iv):
    rng = np.random.default_rng(23)
    n = 8 * nc ** 3
    pos = rng.random((n, 3)) * nc
    pos[: n // 5] = np.array([nc / nnt, 0.1, nc - 0.2]) + 0.4 * rng.standard_normal((n // 5, 3))
    _check(nc, nnt, ncb, ix, iv, np.mod(pos, nc), rng)


def test_coordinate_that_rounds():
    nc = 144
    rng = np.random.default_rng(6)
    cells = np.stack(np.meshgrid(*[np.arange(nc - 16, nc)] * 3, indexing="ij"), -1).reshape(-1, 3)
    c = np.repeat(np.concatenate([cells, rng.integers(0, nc, size=(500, 3))]), 3, axis=0)
    tops = np.array([0, 16383, 16384, 49152, 65535])
    u = np.where(rng.random(c.shape) < 0.7, tops[rng.integers(0, len(tops), c.shape)], rng.integers(0, 65536, c.shape))
    tempx = (4 * c + (u + 0.5) / 16384.0).astype(np.float32)
    assert (np.floor(tempx) == 4 * c + 4).sum() > 1000  # rounded past their cell
    _check(nc, 1, 6, 2, 2, c + (u + 0.5) / 65536.0, rng)
