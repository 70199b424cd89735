"""The kernels' exponential of negative arguments, compiled for the host and held against extended precision.

What it computes goes into products that are within a few units of a rounding boundary, so that a coefficient lost on the way
would show in no bfloat16 result of a random product.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

HIP = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "yvex_amd", "csrc", "hip")
SOURCE = r"""
#include <cfloat>
#include <cmath>
#include "exp_negative.hpp"
// largest distance from the exponential in units of the last place of it in binary64 (of a subnormal's below the normal numbers)
extern "C" double worst(const double *x, long n)
{
    long double most = 0.0L;
    for (long i = 0; i < n; ++i) {
        const long double want = expl((long double)x[i]);
        int exponent = 0;
        frexpl(want, &exponent);
        const int last = exponent - 53 < -1074 ? -1074 : exponent - 53;
        const long double off = fabsl((long double)yvex::exp_of_negative(x[i]) - want) / ldexpl(1.0L, last);
        if (!(off <= most)) most = off;
    }
    return (double)most;
}
"""


@pytest.fixture(scope="module")
def worst(tmp_path_factory):
    import ctypes as C
    compiler = shutil.which("g++")
    if not compiler or np.finfo(np.longdouble).nmant < 63:
        pytest.skip("needs g++ and an 80-bit long double")
    folder = tmp_path_factory.mktemp("exponential")
    source, library = folder / "worst.cpp", folder / "worst.so"
    source.write_text(SOURCE)
    subprocess.run([compiler, "-O2", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off", "-w", "-D__device__=",
                    "-D__forceinline__=inline", f"-I{HIP}", str(source), "-o", str(library)], check=True)
    handle = C.CDLL(str(library))
    handle.worst.restype = C.c_double
    handle.worst.argtypes = [C.c_void_p, C.c_long]
    return lambda x: handle.worst(np.ascontiguousarray(x, dtype=np.float64).ctypes.data, len(x))


# (random arguments, arguments around the middles between multiples of ln 2, where the polynomial's argument is largest, and
# around the multiples; what float32 gates give)
def test_normal_results_are_within_six_tenths_of_a_unit(worst):
    rng = np.random.default_rng(3)
    steps = np.arange(0, 1021)[:, None] * np.log(2.0)
    near = np.concatenate([(-(steps + at) + rng.uniform(-1e-3, 1e-3, (1021, 400))).reshape(-1) for at in (0.0, np.log(2.0) / 2)])
    spread = np.concatenate([-rng.uniform(0.0, 708.0, 1_000_000), -np.exp(rng.uniform(-40.0, np.log(708.0), 1_000_000))])
    gates = -np.abs(rng.standard_normal(500_000) * 8.0).astype(np.float32).astype(np.float64)
    for x in (near[(near <= 0.0) & (near >= -708.0)], spread, gates):
        assert worst(x) <= 0.60
    assert worst(np.array([0.0, -0.0])) == 0.0


# (rounded to 53 bits and again to the subnormal's place: half a unit, and the 0.6 of a unit that is at most half as large)
def test_subnormal_results_and_zero(worst):
    rng = np.random.default_rng(4)
    assert worst(-rng.uniform(708.5, 746.0, 500_000)) <= 0.80
    assert worst(np.array([-745.2, -746.0, -799.0, -801.0, -1e5, -3e38, -np.inf])) <= 0.5
