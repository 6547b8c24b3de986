"""PP on a box with one cell of 10000 particles: some 40 work items of
milliseconds each, fewer than CUs.  Each has a CU of its own, whatever runs
beside PP, so passes take alike; two of them on one CU took 1.3 times as long,
and in the step loop most passes had two that met."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_long_items_do_not_meet_on_a_cu():
    from cafproject_amd.cube import Cube
    nc = 32
    rng = np.random.default_rng(nc)
    x = rng.random((nc ** 3, 3)) * nc
    x[:10000] = nc / 2 + 0.3 + 0.1 * rng.standard_normal((10000, 3))
    v = (0.05 * rng.standard_normal(x.shape)).astype(np.float32)
    g = Cube(nc, 1, np_nc=1, izipx=1, izipv=2, pp_on=True, image_buffer=60.0, tile_buffer=60.0)
    g.init_kernels()
    s = g.set_state_xv(x, v)
    took = []
    for k in range(19):
        t = time.perf_counter()
        g.ext_pp_force(0.1, 1e-6, s, 0.75)
        if k > 3:
            took.append(time.perf_counter() - t)
        g.particle_mesh(0.1, 1e-6, s, s, 0.75)
    took.sort()
    print(" ".join(f"{1e3 * t:.2f}" for t in took))
    assert took[len(took) // 2] < 1.15 * took[0]
