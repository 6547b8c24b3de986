"""The velocity encode of the drift, the kicks and the initial conditions takes
a short atan unless the code is close to a half-integer.  Its codes are the
formula's: on the CPU over the whole range and around every boundary between
two codes, and on the GPU through an initial state around the boundaries."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("enc") / "encode_check.so")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                    os.path.join(HERE, "encode_check.c"), "-o", so, "-lm"], check=True)
    h = ctypes.CDLL(so)
    h.bad_span.argtypes = [ctypes.c_int] + [ctypes.c_double] * 3 + [ctypes.c_int64]
    h.bad_boundaries.argtypes = h.bad_special.argtypes = [ctypes.c_int, ctypes.c_double]
    h.bad_span.restype = h.bad_boundaries.restype = h.bad_special.restype = ctypes.c_int64
    h.worst_y.argtypes, h.worst_y.restype = [ctypes.c_int64], ctypes.c_double
    return h


@pytest.mark.parametrize("bytes_", [1, 2])
def test_codes_on_the_cpu(lib, bytes_):
    for c in (1.0, 0.037, 411.7):
        assert lib.bad_span(bytes_, c, 1e-9, 1e9, 1_000_000) == 0
        assert lib.bad_boundaries(bytes_, c) == 0
        assert lib.bad_special(bytes_, c) == 0


def test_margin_covers_the_fit(lib):
    # 1.4e-10 of the fit in units of the code, with the rest well inside 2^-17
    assert lib.worst_y(2_000_000) < 3e-6


@pytest.mark.gpu
@pytest.mark.parametrize("iv", [1, 2])
def test_codes_on_the_gpu(iv):
    from cafproject_amd import ics
    from cafproject_amd.cube import Cube
    nc, sig = 32, 0.31
    c = float(np.float32(np.sqrt(np.float32(ics.PI_F / 2)))) / (float(np.float32(sig)) * 2.5)
    nvm1 = (1 << (8 * iv)) - 1
    rng = np.random.default_rng(3)
    # two particles a cell with v and -v: the mean is 0 exactly, both codes are of floats at a boundary
    k = (rng.integers(0, nvm1 // 2, size=(nc ** 3, 3)) + 0.5) * ics.PI_F / nvm1
    v = (np.tan(k) / c).astype(np.float32)
    v = np.stack([v, -v], 1).reshape(-1, 3)
    cell = np.stack(np.meshgrid(*[np.arange(nc)] * 3, indexing="ij"), -1).reshape(-1, 1, 3)
    x = (cell + np.array([[[0.25] * 3, [0.75] * 3]])).reshape(-1, 3).astype(np.float64)
    g = Cube(nc, 2, ncb=6, np_nc=2, izipx=2, izipv=iv)
    g.set_state_xv(x, v, sig)
    st = g.get_state()
    ref = ics.encode_v(iv, v, sig).astype(np.int64)
    got = np.empty_like(ref)
    got[st["pid"] - 1] = st["vp"]
    # numpy's atan against the formula's: a code off by one only within 1e-9 of a half-integer
    y = nvm1 * np.arctan(c * v.astype(np.float64)) / ics.PI_F
    near = np.abs(np.abs(y - np.trunc(y)) - 0.5) < 1e-9
    assert np.array_equal(got[~near], ref[~near])
    assert near.mean() < 0.05  # one in 127 boundaries may be a float
