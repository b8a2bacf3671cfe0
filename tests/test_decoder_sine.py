"""The sine of the fused residual units (csrc/decoder.hip, dec_sin2), compiled
for the host: no further from sin^2 than the square of a correctly rounded
sine, in the mean and at the worst argument, over SnakeBeta's range; the
argument's infinities and NaN."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from conftest import PKG


@pytest.fixture(scope="module")
def sin2(tmp_path_factory):
    src = open(os.path.join(PKG, "csrc", "decoder.hip")).read()
    body = re.search(r"__device__ __forceinline__ (float dec_sin2\(float t\) \{\n.*?\n\}\n)", src, re.S).group(1)
    d = tmp_path_factory.mktemp("sine")
    (d / "s.cpp").write_text("#include <cmath>\nstatic " + body + 'extern "C" void run(const float *t, float *o, int n) '
                             "{ for (int i = 0; i < n; i++) o[i] = dec_sin2(t[i]); }\n")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-fPIC", "-shared", str(d / "s.cpp"), "-o", str(d / "s.so")],
                   check=True)
    lib = C.CDLL(str(d / "s.so"))

    def run(t):
        out = np.empty_like(t)
        lib.run(t.ctypes.data_as(C.c_void_p), out.ctypes.data_as(C.c_void_p), t.size)
        return out

    return run


@pytest.mark.parametrize("scale", [0.1, 1.0, 6.0, 300.0, 3000.0])
def test_no_further_than_a_rounded_sine(sin2, scale):
    t = (scale * np.random.default_rng(5).standard_normal(1 << 19)).astype(np.float32)
    s = np.sin(t.astype(np.float64))
    rounded = s.astype(np.float32)
    err, ref = (np.abs(v.astype(np.float64) - s * s) for v in (sin2(t), rounded * rounded))
    # (1.02 for the sine's own terms at small arguments; the library's is 1.03 to 1.17)
    assert np.sqrt(np.mean(err ** 2)) <= 1.02 * np.sqrt(np.mean(ref ** 2))
    # half an ulp of the sine twice and of the square once is 1.5 * 2^-24 of a
    # square below 1, and the sine's own terms take 2^-26 more
    assert err.max() <= 1.75 * 2.0 ** -24
    # relative to the square: 2^-24 each from the last two roundings of the
    # sine (twice) and of the square, and 0.35 * 2^-24 (twice) from the sine's
    # polynomial.  Past some 50 periods the argument's reduction leaves more
    # near a multiple of pi, of squares below 1e-10.
    if scale <= 6.0:
        nz = s != 0
        assert np.all(err[nz] <= 3.7 * 2.0 ** -24 * (s[nz] * s[nz]))


def test_not_finite(sin2):
    assert np.all(np.isnan(sin2(np.array([np.inf, -np.inf, np.nan], dtype=np.float32))))
    assert np.array_equal(sin2(np.array([0.0, -0.0], dtype=np.float32)), [0.0, 0.0])
