"""The limiter's least ratio with two divisions (anuga_core_amd/csrc/
de_limit.h), compiled for the host, against limit_gradient's sequence of
three: the same values for jumps of both signs, equal ones, zeros and jumps at
the threshold, bounds that are zero, infinities and NaN."""

import ctypes as C
import itertools
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "anuga_core_amd", "csrc")
SOURCE = r"""
#include "de_limit.h"
extern "C" void ratios(long n, const double *d, const double *q, double *two, double *three)
{
    for (long k = 0; k < n; k++, d += 3, q += 2) {
        two[k] = de_limit_ratio(d, q[0], q[1]);
        double r = 1000.0, r0 = 1.0;
        for (int i = 0; i < 3; i++) {
            if (d[i] < -1.0e-100) r0 = q[0] / d[i];
            if (d[i] > 1.0e-100) r0 = q[1] / d[i];
            r = fmin(r0, r);
        }
        three[k] = r;
    }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    tmp = tmp_path_factory.mktemp("limiter")
    src, so = tmp / "limiter.cpp", tmp / "liblimiter.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC",
                    "-I" + CSRC, "-o", str(so), str(src)], check=True)
    return C.CDLL(str(so))


@pytest.mark.parametrize("kind", ["random", "scales", "special"])
def test_two_divisions_give_the_values_of_three(lib, kind):
    rng = np.random.default_rng(2)
    if kind == "special":
        v = [0.0, -0.0, 1.0e-100, -1.0e-100, 1.1e-100, -1.1e-100, 5.0e-324, 0.3, -0.3, 0.7, 1e300,
             -1e300, np.inf, -np.inf, np.nan]
        d = np.array(list(itertools.product(v, v, v)))
        lo, hi = [0.0, -0.0, -0.2, -5e-324, -1e300, -np.inf], [0.0, 0.3, 1e-320, 1e300, np.inf]
        q = np.array(list(itertools.product(lo, hi)))
        d, q = np.repeat(d, len(q), axis=0), np.tile(q, (len(d), 1))
    else:
        n = 300000
        d, q = rng.standard_normal((n, 3)), rng.standard_normal((n, 2))
        if kind == "scales":
            d *= 10.0 ** rng.integers(-110, 5, (n, 3))
            q *= 10.0 ** rng.integers(-110, 5, (n, 2))
            d[::5, 1] = d[::5, 0]
            d[::7, 0] = 0.0
        else:
            d[:, 2] = np.where(rng.random(n) < 0.3, np.nextafter(d[:, 0], 9.0), d[:, 2])
        q = np.stack([-np.abs(q[:, 0]), np.abs(q[:, 1])], axis=1)
    d, q = np.ascontiguousarray(d), np.ascontiguousarray(q)
    two, three = np.zeros(len(d)), np.zeros(len(d))
    dp = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))
    lib.ratios(C.c_long(len(d)), dp(d), dp(q), dp(two), dp(three))
    assert not np.isnan(three).any()
    assert np.array_equal(two, three)
