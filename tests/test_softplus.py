"""csrc/kh_softplus.h, the code that the kernels run, compiled for the host, against 64 bits."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "kuiperllama_amd", "csrc")
SRC = """#include "kh_softplus.h"
extern "C" void softplus(const float* z, float* o, long n, float off) {
  for (long i = 0; i < n; ++i) o[i] = softplus_of(z[i], [=](float h) { return 1.0f / h * off; });
}
"""


@pytest.fixture(scope="module")
def softplus(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("softplus")
    (d / "s.cpp").write_text(SRC)
    subprocess.check_call([cxx, "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", "-I", CSRC, str(d / "s.cpp"), "-o", str(d / "s.so")])
    f = ctypes.CDLL(str(d / "s.so")).softplus
    f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_long, ctypes.c_float]

    def run(z, off=1.0):
        z = np.ascontiguousarray(z, np.float32)
        o = np.empty_like(z)
        f(z.ctypes.data, o.ctypes.data, z.size, off)
        return o
    return run


# the hardware's reciprocal is within one unit in the last place
@pytest.mark.parametrize("off", [1.0, 1.0 + 2.0 ** -23, 1.0 - 2.0 ** -24])
@pytest.mark.parametrize("lo,hi", [(-104, -87.3), (-87.3, -30), (-30, -8), (-8, -3), (-3, -1), (-1, 0), (0, 1), (1, 3), (3, 8), (8, 30), (30, 200)])
def test_error_against_64_bits(softplus, lo, hi, off):
    """Below one unit in the last place (of a denormal result: of the smallest): 1/2 from the last rounding, 1/4 from the first
    term that the series leaves out ((1/9)^7 / 15 at z = 0), and 1/5 from a remainder of s of up to 1.5 units that is added
    without its factor of at most 9/8."""
    z = np.random.default_rng(3).uniform(lo, hi, 1 << 15).astype(np.float32)
    x = z.astype(np.float64)
    want = np.maximum(x, 0.0) + np.log1p(np.exp(-np.abs(x)))
    unit = np.maximum(np.spacing(want.astype(np.float32)).astype(np.float64), 2.0 ** -149)
    assert np.all(np.abs(softplus(z, off) - want) < unit)


def test_edges(softplus):
    z = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 3e38, -3e38, 1e-40], np.float32)
    got = softplus(z)
    ln2 = np.float32(np.log(2.0))
    np.testing.assert_array_equal(got[[0, 1, 7]], ln2)
    assert got[2] == np.inf and got[3] == 0.0 and np.isnan(got[4]) and got[5] == np.float32(3e38) and got[6] == 0.0
