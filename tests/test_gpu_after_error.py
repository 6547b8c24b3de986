"""A call that a HIP error ends between two of its kernels leaves nothing behind
that the next call takes for its own.  The error is one that an earlier, refused
HIP call left unread (a device number that does not exist): the library reports
it at its first launch, which here is the fine deposit's kernel that lists the
blocks with crowded cells (CUBE_FD_HEAVY=0: every block), and the kernel that
empties the list is never queued.  The same call again equals a new context's,
and the calls after it too."""
import numpy as np
import pytest

from tests.helpers import zeldovich_state

pytestmark = pytest.mark.gpu

A, DT = 0.1, 4.0


def _cube(st):
    from cafproject_amd.cube import Cube
    g = Cube(24, 2)
    g.init_kernels()
    g.set_state(st["xp"], st["vp"], st["pid"], st["rhoc"], st["vfield"])
    return g


def _fail(call):
    from cafproject_amd.cube import CubeError, lib
    assert lib().hipSetDevice(1 << 20) != 0  # refused by the runtime; the error stays to be read
    with pytest.raises(CubeError) as e:
        call()
    assert e.value.code == 10


@pytest.mark.parametrize("times", [1, 3])
def test_calls_after_a_failed_one(times, monkeypatch):
    monkeypatch.setenv("CUBE_FD_HEAVY", "0")
    st = zeldovich_state(24, 2, seed=5)
    s, m = st["sigma_vi"], 0.75
    ref, g = _cube(st), _cube(st)
    for _ in range(times):
        _fail(lambda: g.fine_deposit(m))
    assert g.fine_deposit(m) == ref.fine_deposit(m)
    assert np.array_equal(g.get_field("rho_f"), ref.get_field("rho_f"))
    for _ in range(times):
        _fail(lambda: g.particle_mesh(A, DT, s, s, m))
    for _ in range(2):  # the second step finds the words as the first left them
        a, b = g.particle_mesh(A, DT, s, s, m), ref.particle_mesh(A, DT, s, s, m)
        assert all(np.array_equal(a[k], b[k]) for k in b)
        assert np.array_equal(g.get_state()["vp"], ref.get_state()["vp"])
