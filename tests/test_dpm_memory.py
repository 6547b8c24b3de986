"""Force meshes that a box of the differentiable model keeps for its adjoint do
not take the room of boxes made later: of every size, as many boxes as fill a
device at the memory that they took with their deposits in 64-bit meshes (30
bytes per mesh point and 36 per particle more, and no force meshes kept) still
fit, and a few boxes have theirs."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
GB = 1 << 30


@pytest.fixture(scope="module")
def boxes(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("mem") / "dpm_memory_check.so")
    subprocess.run(["gcc", "-O2", "-shared", "-fPIC", os.path.join(HERE, "dpm_memory_check.c"), "-o", so], check=True)
    f = ctypes.CDLL(so).boxes
    f.argtypes = [ctypes.c_uint64] * 3 + [ctypes.c_int64] * 2 + [ctypes.POINTER(ctypes.c_int64)]
    f.restype = ctypes.c_int64

    def run(total, base, extra, nf3, np_):
        kept = ctypes.c_int64()
        return f(total, base, extra, nf3, np_, ctypes.byref(kept)), kept.value
    return run


@pytest.mark.parametrize("ng,nf", [(32, 64), (96, 96), (96, 192), (128, 256), (64, 256), (256, 512)])
@pytest.mark.parametrize("nsteps", [1, 2, 10, 18, 40, 155, 400])
def test_as_many_boxes_fit(boxes, ng, nf, nsteps):
    nf3, np_ = nf ** 3, ng ** 3
    # meshes: density, force, cotangents, lambda, 1 + 3 half spectra; particles:
    # positions of all steps, momenta, two cotangents; tile lists up to 14 bytes;
    # amplitude, noise spectra and displacement planes of the lattice
    base = int(48.5 * nf3 + (12 * (nsteps + 1) + 36 + 14 + 30.5) * np_)
    for total in (288 * GB, 48 * GB):
        n, kept = boxes(total, base, 12 * (nsteps - 1) * nf3, nf3, np_)
        assert n >= total // (base + 30 * nf3 + 36 * np_)
        assert kept * 12 * (nsteps - 1) * nf3 <= total // 4
        if nsteps == 10 and total == 288 * GB:
            assert kept >= 1
    if (ng, nf, nsteps) == (128, 256, 10):
        print(boxes(288 * GB, base, 12 * 9 * nf3, nf3, np_))
