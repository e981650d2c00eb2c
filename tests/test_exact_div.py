"""xdiv (mdoodz7.0_amd/csrc/exact_div.h), the division by a cell width of the
marker kernels, is the IEEE division bit for bit: the header compiled for
the host against a / b over cell widths and marker distances, significands
next to powers of two and to each other (where a quotient is hardest to
round), the ends of the accepted exponent range and what lies beyond it
(zeros, infinities, NaN, subnormal and extreme values, extreme divisors)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT

SRC = r"""
#include "exact_div.h"
using std::fma;
extern "C" void run(long n, const double *a, double b, double *q) {
    const exact_div d = make_exact_div(b);
    for (long i = 0; i < n; i++) q[i] = xdiv(a[i], d);
}
"""


@pytest.fixture(scope="module")
def div(tmp_path_factory):
    p = tmp_path_factory.mktemp("xdiv")
    (p / "x.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "mdoodz7.0_amd", "csrc"), str(p / "x.cpp"), "-o", str(p / "x.so")],
                   check=True)
    f = ctypes.CDLL(str(p / "x.so")).run
    f.argtypes = [ctypes.c_long, ctypes.c_void_p, ctypes.c_double, ctypes.c_void_p]

    def run(a, b):
        a = np.ascontiguousarray(a)
        q = np.empty_like(a)
        f(a.size, a.ctypes.data, float(b), q.ctypes.data)
        with np.errstate(all="ignore"):
            ref = a / np.float64(b)
        nan = np.isnan(ref)
        assert np.array_equal(nan, np.isnan(q))
        assert np.array_equal(q.view(np.uint64)[~nan], ref.view(np.uint64)[~nan]), b
    return run


def _near(rng, n):
    """Significands a few units from powers of two and from simple fractions."""
    m = np.ldexp(1.0, rng.integers(-40, 40, n)) * rng.choice([1.0, 1.5, 4 / 3, 1.25, 2 - 2 ** -52], n)
    return (m.view(np.int64) + rng.integers(-8, 9, n)).view(np.float64)


def test_marker_distances(div):
    rng = np.random.default_rng(5)
    for h in [1 / 2047, 1 / 101, 1e6 / 4095, 250e3 / 1023, 0.1, 1.0, 3.0, 1 / 3, 2 - 2 ** -52, 1 + 2 ** -52] + \
            list(rng.uniform(1e-6, 1e4, 40)) + list(_near(rng, 40)):
        d = rng.uniform(-2, 3000, 4000) * h
        v = rng.standard_normal(4000) * rng.uniform(0, 1, 4000) * h
        k = rng.integers(0, 3000, 4000).astype(float) * h             # on cell edges
        div(np.concatenate([d, v, k, np.nextafter(k, 0), np.nextafter(k, 1e9), _near(rng, 4000), -_near(rng, 4000)]), h)


def test_beyond_the_range(div):
    rng = np.random.default_rng(6)
    e = np.concatenate([np.arange(-1074, -1010), np.arange(-520, -500), np.arange(500, 524), np.arange(1000, 1024)])
    a = np.ldexp(rng.uniform(1, 2, e.size), e)
    a = np.concatenate([a, -a, [0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, 1.7976931348623157e308]])
    for b in (1.0, 1 / 3, 1e-3, 2.0 ** 128, 2.0 ** -128, 1e-39, 1e39, 1e-300, 1e300, 5e-324, np.inf, 0.0, -0.7):
        div(a, b)
