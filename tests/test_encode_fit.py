"""The velocity encode decides a code by a short atan unless the value lies
within 2^-17 of a half-integer.  That is sound while the fit in the library is
off by less: its error over (0, 1], in units of the 2-byte code, is measured
here on the library's own polynomial and stays under 3e-6, which leaves room
for the roundings (3e-11) and the reciprocal (2^-44 of 16384 codes, 1e-9)."""
import ctypes
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_margin_covers_the_library_s_fit(tmp_path):
    so = str(tmp_path / "atan_fit_check.so")
    subprocess.run(["gcc", "-O2", "-mfma", "-ffp-contract=off", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                    os.path.join(HERE, "atan_fit_check.c"), "-o", so, "-lm"], check=True)
    f = ctypes.CDLL(so).worst_fit
    f.argtypes, f.restype = [ctypes.c_int64], ctypes.c_double
    worst = f(2_000_000)
    assert 1e-7 < worst < 3e-6 < 2.0 ** -17
