"""The Green's function pass at every small mesh size, where its work is split
over line sets and components, with three force spectra and with one: the fine
and coarse forces of a random density against the FP64 transform of the same
density with the library's own kernels.  An FP32 transform pair errs by some 2
log2(N^3) roundings of 2^-24, 3e-6 for the largest here."""
import numpy as np
import pytest

from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu


def _force(rho, K):
    n = rho.shape[0]
    sp = np.fft.rfftn(rho.astype(np.float64))
    return np.stack([np.fft.irfftn(1j * K[d] * sp, s=(n, n, n), axes=(0, 1, 2)) for d in range(3)], -1)


@pytest.mark.parametrize("layout", [1, 2])
@pytest.mark.parametrize("nc", [12, 16, 18, 20, 24, 32, 48])
def test_forces(nc, layout):
    from cafproject_amd.cube import Cube
    nf, h = 4 * nc, 2 * nc
    rng = np.random.default_rng(nc)
    g = Cube(nc, 1, np_nc=1, mem_layout=layout)
    g.init_kernels()
    rho = rng.random((nf,) * 3, dtype=np.float32) * 2
    g.set_field("rho_f", rho)
    g.fine_force()
    o = g.get_field("kern_f").astype(np.float64)  # octant, odd in k_d
    k = np.arange(nf)
    kk, s = np.where(k <= h, k, nf - k), np.where(k <= h, 1.0, -1.0)
    full = o[:, kk][:, :, kk]
    full[1] *= s[None, :, None]
    full[2] *= s[:, None, None]
    assert rel_l2(g.get_field("force_f"), _force(rho, full)) < 1e-5
    rho = rng.random((nc,) * 3, dtype=np.float32) * 2
    g.set_field("rho_c", rho)
    g.coarse_force()
    assert rel_l2(g.get_field("force_c"), _force(rho, g.get_field("kern_c").astype(np.float64))) < 1e-5
