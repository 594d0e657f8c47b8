"""The FP64 exp, log and reciprocal of the z-node arithmetic (threepoint_amd/csrc/tp_fp64.h), built by the host
compiler and (gpu) in a kernel, against 80-bit arithmetic.  The bounds follow from the forms: exp is a degree-11 polynomial whose last
step rounds once at 0.5 ulp over an argument reduction good to 2^-56 and inner steps weighted by |r| < 0.35
(< 1 ulp together); the reciprocal's third-order step leaves its cubed seed error and one rounding (< 1 ulp); exp10 is
exp and the rounding of its remainder's product (< 1.5 ulp).  log ends in one rounded addition (0.5 ulp), and what is added to the exact
k ln 2 - ln c carries the roundings of r and of the sum q (2^-62 each, both below 2^-8), the table's residual (0.56 2^-62)
and the series' remainder (0.64 2^-62): below 2^-60 absolute together; log1p adds one more rounding of the sum."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "tp_fp64.h"
#include <cstdio>
#include <cmath>
extern "C" void run(int what, int n, const double *x, double *y, long double *ref)
{
    for (int i = 0; i < n; ++i) {
        if (what == 0) { y[i] = tp_fp64_exp(x[i]); if (ref) ref[i] = expl(x[i]); }
        else if (what == 1) { y[i] = tp_fp64_log(x[i]); if (ref) ref[i] = logl(x[i]); }
        else if (what == 2) { y[i] = tp_fp64_rcp(x[i]); if (ref) ref[i] = 1.0L / x[i]; }
        else if (what == 3) { y[i] = tp_fp64_log1p(x[i]); if (ref) ref[i] = log1pl(x[i]); }
        else if (what == 4) { y[i] = tp_fp64_exp10(x[i]); if (ref) ref[i] = powl(10.0L, x[i]); }
        else if (what == 5) { y[i] = tp_fp64_exp_any(x[i]); if (ref) ref[i] = expl(x[i]); }
        else if (what == 6) { y[i] = tp_fp64_exp_low(x[i]); if (ref) ref[i] = expl(x[i]); }
        else { y[i] = tp_fp64_rcp_any(x[i]); if (ref) ref[i] = 1.0L / x[i]; }
    }
}
"""


@pytest.fixture(scope="module")
def fp64(tmp_path_factory):
    import ctypes
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("fp64")
    (d / "t.cpp").write_text(SRC)
    subprocess.run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC", "-ffp-contract=off",
                    "-I" + os.path.join(ROOT, "threepoint_amd", "csrc"), str(d / "t.cpp"), "-o", str(d / "t.so")],
                   check=True)
    lib = ctypes.CDLL(str(d / "t.so"))

    def call(what, x):
        x = np.ascontiguousarray(x, dtype=np.float64)
        y, ref = np.zeros(x.size), np.zeros(x.size, dtype=np.longdouble)
        lib.run(what, x.size, x.ctypes.data_as(ctypes.c_void_p), y.ctypes.data_as(ctypes.c_void_p),
                ref.ctypes.data_as(ctypes.c_void_p))
        return y, ref
    return call


def _ulps(y, ref, absolute=0.0):
    """Largest error in ulps, after an absolute allowance."""
    r = np.maximum(np.abs(ref).astype(np.float64), np.finfo(float).tiny)
    return np.max(np.maximum(np.abs(y.astype(np.longdouble) - ref) - absolute, 0) / np.spacing(r))


def _samples(what):
    rng = np.random.default_rng(11 + what)
    if what == 0:  # every scale down to 0, and the whole range of normal results
        x = np.concatenate([rng.uniform(-700, 700, 200000), rng.uniform(-40, 40, 200000),
                            rng.choice([-1, 1], 100000) * np.exp(rng.uniform(-40, 3, 100000)),
                            np.arange(-1000, 1001) * (0.5 * np.log(2.0))])
        x = x[np.abs(x) < 700]
    elif what == 1:  # all binades, and both sides of 1 and of sqrt(1/2), the table's interval ends
        x = np.concatenate([np.exp(rng.uniform(-700, 700, 200000)), 1 + rng.uniform(-1, 1, 200000) * 0.5,
                            np.sqrt(0.5) * (1 + rng.uniform(-1, 1, 50000) * 1e-6), np.exp(rng.uniform(1, 12, 200000)),
                            [np.finfo(float).tiny, np.finfo(float).max, 0.5, 2.0],
                            2.0 ** rng.integers(-1000, 1000, 500) * (1 + np.arange(500) % 129 / 128.0)])
    elif what == 2:
        x = rng.choice([-1, 1], 400000) * np.exp(rng.uniform(-700, 700, 400000))
    elif what == 3:
        x = np.concatenate([np.exp(rng.uniform(-100, 100, 400000)), rng.uniform(0, 3, 100000), [0.0, 1.0, 1e-300]])
    else:
        x = np.concatenate([rng.uniform(-300, 300, 200000), rng.uniform(-8, 8, 200000), np.arange(-300.0, 301.0)])
    return x


FORMS = [(0, 1.0), (1, 0.51), (2, 1.0), (3, 1.01), (4, 1.5)]


@pytest.mark.parametrize("what, bound", FORMS)
def test_errors(fp64, what, bound):
    x = _samples(what)
    y, ref = fp64(what, x)
    u = _ulps(y, ref, 2.0 ** -60 if what in (1, 3) else 0.0)
    print("what %d: max error %.3f ulp of %d" % (what, u, x.size))
    assert u < bound


def test_ends_of_the_range(fp64):
    y, _ = fp64(0, [800.0, 5000.0, -800.0, -5000.0, 0.0, np.nan])
    assert np.all(np.isinf(y[:2])) and np.all(y[2:4] == 0) and y[4] == 1 and np.isnan(y[5])
    y, _ = fp64(1, [1.0])
    assert abs(y[0]) < 2.0 ** -60


def test_the_whole_stated_domain_and_the_forms_for_any_argument(fp64):
    """exp up to 2^30 either way; exp_any and exp_low beyond it, infinities included, and rcp_any at the infinities,
    each with the bits of the plain form inside its range."""
    far = np.array([1e4, 1.4e9 / 2, 2.0 ** 30])
    y, _ = fp64(0, np.concatenate([far, -far]))
    assert np.all(np.isposinf(y[:3])) and np.all(y[3:] == 0)
    farther = np.array([1.4e9, 1.5e9, 2.0 ** 31 - 1, 2.1e9, 1e10, 1e15, 1e18, 1e100, 1e300, np.inf])
    assert np.all(np.isposinf(fp64(5, farther)[0])) and np.all(fp64(5, -farther)[0] == 0)
    assert np.all(fp64(6, -farther)[0] == 0)
    y, _ = fp64(7, [np.inf, -np.inf, np.nan])
    assert y[0] == 0 and not np.signbit(y[0]) and y[1] == 0 and np.signbit(y[1]) and np.isnan(y[2])
    x = np.random.default_rng(3).uniform(-700, 700, 20000)
    for form, plain in ((5, 0), (6, 0), (7, 2)):
        assert np.array_equal(fp64(form, x)[0], fp64(plain, x)[0])
    e = np.exp(np.random.default_rng(4).uniform(-700, 700, 20000))
    assert np.array_equal(fp64(7, e)[0], fp64(2, e)[0])


def _device(what, x):
    import ctypes
    lib = ctypes.CDLL(os.path.join(ROOT, "tests", "fp64_device", "_build", "fp64_device.so"))
    x = np.ascontiguousarray(x, dtype=np.float64)
    y = np.zeros(x.size)
    assert lib.run(what, x.size, x.ctypes.data_as(ctypes.c_void_p), y.ctypes.data_as(ctypes.c_void_p)) == 0
    return y


@pytest.mark.gpu
@pytest.mark.parametrize("what, bound", FORMS)
def test_errors_on_the_device(what, bound):
    """The forms as a kernel contains them, on the samples and to the bounds of the host build."""
    x = _samples(what)
    v = x.astype(np.longdouble)
    ref = [np.exp, np.log, lambda t: 1 / t, np.log1p, lambda t: np.longdouble(10) ** t][what](v)
    u = _ulps(_device(what, x), ref, 2.0 ** -60 if what in (1, 3) else 0.0)
    print("what %d: max error %.3f ulp of %d" % (what, u, x.size))
    assert u < bound


@pytest.mark.gpu
def test_ends_of_the_range_on_the_device():
    """The range's ends and the forms for any argument, as in the host build."""
    y = _device(0, [800.0, 2.0 ** 30, -800.0, -2.0 ** 30, 0.0, np.nan])
    assert np.all(np.isposinf(y[:2])) and np.all(y[2:4] == 0) and y[4] == 1 and np.isnan(y[5])
    far = np.array([1.5e9, 2.0 ** 31 - 1, 2.1e9, 1e15, 1e100, 1e300, np.inf])
    assert np.all(np.isposinf(_device(5, far))) and np.all(_device(5, -far) == 0) and np.all(_device(6, -far) == 0)
    y = _device(7, [np.inf, -np.inf, np.nan, 1.0, -4.0])
    assert y[0] == 0 and not np.signbit(y[0]) and y[1] == 0 and np.signbit(y[1]) and np.isnan(y[2])
    assert y[3] == 1 and y[4] == -0.25
    x = _samples(2)
    assert np.array_equal(_device(7, x), _device(2, x))
