"""The drift's finalize pass at the edges of its runs: cells at, below and above
the 64 keys that it ranks in LDS, the 640 slots of a run and the 1024 and 16384
keys of the sorts for larger ones, side by side in one workgroup's 64 cells,
with empty cells between.  Bit for bit against the oracle."""
import numpy as np
import pytest

from cafproject_amd import ics
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[0, 640, 0, 1, 63, 64, 65, 0, 2, 641, 5, 1, 0, 1279, 1280, 1281, 3],
                                    [1024, 1025, 0, 0, 64, 64, 64, 64, 64, 64, 64, 64, 64, 64, 64, 1, 66],
                                    [16384, 1, 16385, 0, 70], []])
@pytest.mark.parametrize("ix,iv", [(1, 2), (2, 1)])
def test_runs_of_cells(counts, ix, iv):
    from cafproject_amd.cube import Cube
    nc, nnt = 16, 2
    nt = nc // nnt
    rng = np.random.default_rng(17)
    n = np.full(nc ** 3, 0)
    n[64 * 5:64 * 5 + len(counts)] = counts  # in disjoint order: within finalize workgroup 5
    n[64 * 9:64 * 20] = rng.integers(0, 24, 64 * 11)  # some workgroups above 640 slots, some below
    cid = np.repeat(np.arange(nc ** 3), n)
    i, j, k, t = cid % nt, (cid // nt) % nt, (cid // nt ** 2) % nt, cid // nt ** 3
    cell = np.stack([i + nt * (t % nnt), j + nt * ((t // nnt) % nnt), k + nt * (t // nnt ** 2)], -1)
    # particles stay in their cells: 0.3 from the faces, moved by less than 0.2
    pos = cell + 0.3 + 0.4 * rng.random(cell.shape)
    v = (0.01 * rng.standard_normal(cell.shape)).clip(-0.03, 0.03).astype(np.float32)
    st = ics.disjoint_state(pos, v, nc, nnt, izipx=ix, izipv=iv)
    assert np.array_equal(st["rhoc"], n)
    np_nc = max(2, int(np.ceil((len(pos) / nc ** 3) ** (1 / 3))))
    oc = O.OracleCube(nc, nnt, np_nc=np_nc, izipx=ix, izipv=iv, tile_buffer=30.0, image_buffer=30.0)
    oc.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    oc.buffer_grid(); oc.buffer_x(); oc.buffer_v()
    g = Cube(nc, nnt, np_nc=np_nc, izipx=ix, izipv=iv, tile_buffer=30.0, image_buffer=30.0)
    g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    s_o, stats = oc.update_x(20.0, 20.0, 0.5, st["sigma_vi"])
    s_g = g.update_x(20.0, 20.0, 0.5, st["sigma_vi"])
    a, b = g.get_state(), oc.get_state()
    assert np.array_equal(a["rhoc"], n)
    for key in ("xp", "vp", "pid", "rhoc", "vfield"):
        assert np.array_equal(a[key], b[key]), key
    assert s_g["nplocal"] == len(pos)
    # sums of at most 2^16 terms >= 0 in FP64, in two orders
    assert abs(s_g["sum_r"] / stats[1] - 1) < 2 * len(pos) * 2.0 ** -53
