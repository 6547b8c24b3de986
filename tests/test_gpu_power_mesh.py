"""cube_power's gathering deposit at the edges of its blocks: meshes that are no
multiple of the block, of 1, 4/3, 2 and 4 cells per coarse cell, boxes a block
reaches round, crowded and empty cells, one- and two-byte positions; and a mesh
coarser than the cells, which is deposited by atomics.  Against the host
analysis in FP64: the same mode counts and |k|, and Delta^2 to the FP32 FFT's
3 log2(ng) roundings of 2^-24 with two decades between bins."""
import numpy as np
import pytest

from cafproject_amd import ics, power

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ix", [1, 2])
@pytest.mark.parametrize("nc,nnt,ncb,ngs", [(24, 2, 6, (12, 24, 32, 48, 96)), (18, 3, 6, (18, 24, 72)),
                                            (20, 4, 5, (20, 80)), (12, 1, 6, (12, 16, 24, 48))])
def test_meshes(nc, nnt, ncb, ngs, ix):
    from cafproject_amd.cube import Cube
    rng = np.random.default_rng(19)
    n = 8 * nc ** 3
    pos = rng.random((n, 3)) * nc
    pos[: n // 6] = np.array([nc - 0.1, 0.2, nc / 2]) + 0.5 * rng.standard_normal((n // 6, 3))
    pos = np.mod(pos, nc)
    st = ics.disjoint_state(pos, np.zeros_like(pos, dtype=np.float32), nc, nnt, izipx=ix, izipv=2, sigma_vi=1.0)
    g = Cube(nc, nnt, ncb=ncb, izipx=ix, izipv=2, image_buffer=30.0, tile_buffer=30.0)
    g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    for ng in ngs:
        k_h, p_h, n_h = power.state_power(st, nc, nnt, ix, 100.0, ng=ng)
        for noalloc in (False, True):
            k_g, p_g, n_g = g.power(ng, 100.0, noalloc=noalloc)
            m = n_h > 0
            assert np.array_equal(n_g, n_h)
            assert np.allclose(k_g[m], k_h[m], rtol=1e-12, atol=0)
            assert np.abs(p_g[m] / p_h[m] - 1).max() < 100 * 3 * np.log2(ng) * 2.0 ** -24, ng
