"""Accuracy of the line kernels' elementary functions (zodipy_amd/csrc/zodi_line_math.hpp).

The header compiles for the host with g++: the same operation sequences and the same tables
(-ffp-contract=off keeps the host from fusing more than the device source asks for).
Errors are measured against mpmath, relative ones of the exact value in units of 2^-53 of
it (an ulp is one to two such units).
"""

from __future__ import annotations

import ctypes as ct
import shutil
import subprocess
from pathlib import Path

import mpmath
import numpy as np
import pytest

CSRC = Path(__file__).resolve().parents[1] / "zodipy_amd" / "csrc"

HARNESS = r"""
#include "zodi_line_math.hpp"
using namespace zodi;
extern "C" void eval(int which, const double* x, double* out, long n) {
  const ExpConst e = exp_const();
  const LogConst l = log_const();
  static double2 log_tab[256];
  for (int j = 0; j < 256; ++j) log_tab[j] = double2{kLineInv[j], kLineLog[j]};
  for (long i = 0; i < n; ++i) {
    switch (which) {
      case 0: out[i] = exp_neg_node(e, x[i]); break;
      case 2: out[i] = exp_neg_cut(e, x[i]); break;
      case 3: out[i] = log_node(log_tab, l, x[i]); break;
      case 4: out[i] = asin_unit(x[i]); break;
      default: out[i] = exp_neg_any(e, x[i]); break;
    }
  }
}
extern "C" void power(double p, double factor, int e_first, double less, const double* x,
                      double* out, long n) {
  static PowTable tab;
  const ExpConst e = exp_const();
  build_pow_table(tab, e, p, factor, e_first, 0, 1);
  const PowPoly q = pow_poly(p);
  for (long i = 0; i < n; ++i)
    out[i] = less == 0.0 ? pow_table(tab, q, x[i]) : pow_table_less(tab, q, x[i], less);
}
extern "C" void angle(int which, const double* x, const double* y, double* out, long n) {
  static AngleTable tab;
  load_angles(tab, 0, 1);
  for (long i = 0; i < n; ++i)
    out[i] = which == 0 ? unit_angle(tab, x[i], y[i]) : axis_angle(x[i], y[i]);
}
"""

P = ct.POINTER(ct.c_double)
EPS = 2.0**-53


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("line_math")
    (d / "harness.cpp").write_text(HARNESS)
    subprocess.run([cxx, "-O2", "-ffp-contract=off", "-std=c++17", "-shared", "-fPIC",
                    f"-I{CSRC}", str(d / "harness.cpp"), "-o", str(d / "lib.so")], check=True)
    return ct.CDLL(str(d / "lib.so"))


def rows(*arrays):
    return [np.ascontiguousarray(a, dtype=np.float64) for a in np.broadcast_arrays(*arrays)]


def ptr(a):
    return a.ctypes.data_as(P)


@pytest.fixture(scope="module")
def fn(lib):
    def f(which, x):
        (x,) = rows(x)
        out = np.empty_like(x)
        lib.eval(which, ptr(x), ptr(out), ct.c_long(x.size))
        return out

    return f


@pytest.fixture(scope="module")
def angle(lib):
    def f(which, x, y):
        x, y = rows(x, y)
        out = np.empty_like(x)
        lib.angle(which, ptr(x), ptr(y), ptr(out), ct.c_long(x.size))
        return out

    return f


@pytest.fixture(scope="module")
def power(lib):
    def f(p, x, factor=1.0, e_first=-100, less=0.0):
        (x,) = rows(x)
        out = np.empty_like(x)
        lib.power(ct.c_double(p), ct.c_double(factor), ct.c_int(e_first), ct.c_double(less),
                  ptr(x), ptr(out), ct.c_long(x.size))
        return out

    return f


def relative(got, exact):
    """|got - exact| / (2^-53 |exact|) for mpmath values, above the subnormal range."""
    return np.array([float(abs((mpmath.mpf(g) - e) / e)) for g, e in zip(got, exact)]) / EPS


@pytest.fixture(autouse=True)
def precision():
    mpmath.mp.prec = 160


@pytest.mark.parametrize("which", [0, 1])
@pytest.mark.parametrize("lo,hi", [(-5.0, 0.0), (0.0, 1.0), (1.0, 10.0), (10.0, 40.0),
                                   (40.0, 200.0), (200.0, 700.0)])
def test_exp(fn, which, lo, hi):
    """Within 2^-53 (1 + 1.3) of the exact value: the table entry and the result are
    rounded (half an ulp, at most 2^-53 each) and the series leaves out 3.8e-17 (0.34);
    the argument's reduction adds nothing that grows with it."""
    x = np.random.default_rng(int(lo + 10) + which).uniform(lo, hi, 4000)
    err = relative(fn(which, x), [mpmath.exp(-mpmath.mpf(v)) for v in x])
    assert err.max() <= 2.4, err.max()
    assert err.mean() <= 0.8, err.mean()


def test_exp_small_arguments(fn):
    """1 - exp(-x), the bands' radial cut-off, keeps its digits: exp is correctly rounded
    next to 1."""
    s = np.concatenate([10.0 ** np.linspace(-12, -3.2, 50), [1e-300, 5e-324, 0.0]])
    for sign in (-1.0, 1.0):
        exact = np.array([float(mpmath.exp(-mpmath.mpf(sign * v))) for v in s])
        np.testing.assert_array_equal(fn(0, sign * s), exact)
        np.testing.assert_array_equal(fn(1, sign * s), exact)
        np.testing.assert_array_equal(fn(2, sign * s), exact)


def test_exp_of_the_cut_off(fn):
    """1 - exp(-x) and x exp(-x) to a rounding of 1 and of the largest x exp(-x)."""
    x = np.random.default_rng(5).uniform(0.0, 38.0, 6000)
    got = fn(2, x)
    exact = [mpmath.exp(-mpmath.mpf(v)) for v in x]
    err = np.array([float(abs(mpmath.mpf(g) - e)) for g, e in zip(got, exact)])
    own = np.array([float(e) for e in exact]) * 2.4 * EPS  # exp's own (test_exp)
    assert np.all(err <= own + 6e-18) and np.all(x * err <= x * own + 8e-18)


def test_exp_ends(fn):
    x = np.array([746.0, 800.0, 5e6, np.nan, -710.0])
    for which in (0, 1):
        got = fn(which, x)
        assert np.all(got[:3] == 0.0) and np.isnan(got[3]) and np.isinf(got[4])
    # past 5.8e6 the exponent's integer saturates
    assert np.all(fn(1, np.array([5.7e6, 5.9e6, 1e12, 1e15, 1e30, 1e90])) == 0.0)


@pytest.mark.parametrize("lo,hi", [(-1.0, 1.0), (-20.0, 10.0), (-100.0, 155.0), (-900.0, 900.0)])
def test_log(fn, lo, hi):
    """Half an ulp of the result, two roundings of values below 1 (the table entry and the
    sum of it and log(1 + r), 2^-54 each) and 1.4e-17 left out of the series."""
    rng = np.random.default_rng(int(hi))
    x = 2.0 ** rng.uniform(lo, hi, 6000)
    got = fn(3, x)
    err = np.array([float(abs(mpmath.mpf(g) - mpmath.log(mpmath.mpf(v)))) for g, v in zip(got, x)])
    bound = 0.5 * np.spacing(np.abs(got)) + 2 * 2.0**-54 + 2e-17
    assert np.all(err <= bound), (err - bound).max()


def test_log_special_values(fn):
    got = fn(3, np.array([np.nan, 2.0, 2.0**-1000]))
    assert np.isnan(got[0]) and abs(got[1] - np.log(2.0)) <= 2.0**-53
    assert abs(got[2] + 1000 * np.log(2.0)) <= np.spacing(1000 * np.log(2.0))


def exact_angle(x, y):
    return [mpmath.atan2(mpmath.mpf(b), mpmath.mpf(a)) for a, b in zip(x, y)]


def directions(seed):
    """Angles over [0, pi], next to both ends, to pi/2 and to the middles between entries."""
    rng = np.random.default_rng(seed)
    th = np.concatenate([rng.uniform(0, np.pi, 4000), 10.0 ** rng.uniform(-12, 0, 500),
                         np.pi - 10.0 ** rng.uniform(-12, 0, 500),
                         np.arange(1, 256) * (np.pi / 256), [0.0, np.pi / 2]])
    return np.cos(th), np.sin(th)


def test_unit_angle(angle):
    """Half an ulp of the angle and the turn's: the direction's two roundings (2^-54 each,
    times c and s), that of the product c sin (2^-54) and of the difference (below 2^-60);
    next to 0 the relative error of s."""
    c, s = directions(1)
    got = angle(0, c, s)
    exact = exact_angle(c, s)
    err = np.array([float(abs(mpmath.mpf(g) - e)) for g, e in zip(got, exact)])
    bound = 0.5 * np.spacing(got) + (np.sqrt(2.0) + 1.0) * 2.0**-54 + 2.0**-59
    assert np.all(err <= bound), (err - bound).max()
    small = got < 0.012
    assert small.sum() > 300
    assert relative(got[small & (s > 0)], [e for e, k in zip(exact, small & (s > 0)) if k]
                    ).max() <= 4.0


def test_unit_angle_ends(angle):
    got = angle(0, np.array([1.0, 0.0, -1.0, np.nan, 0.5]), np.array([0.0, 1.0, 0.0, 0.5, np.nan]))
    assert got[0] == 0.0 and abs(got[1] - np.pi / 2) <= 2.3e-16 and abs(got[2] - np.pi) <= 4.5e-16
    assert np.isnan(got[3:]).all()


def test_axis_angle(angle):
    """As atan2_fast (2 ulp) over vectors of any length."""
    rng = np.random.default_rng(2)
    c, s = directions(3)
    r = 10.0 ** rng.uniform(-6, 3, c.size)
    x, y = c * r, s * r
    got = angle(1, x, y)
    exact = exact_angle(x, y)
    nonzero = np.array([e != 0 for e in exact])
    ulp = np.spacing(np.abs(got))
    err = np.array([float(abs(mpmath.mpf(g) - e)) for g, e in zip(got, exact)])
    assert np.all(err[nonzero] <= 2.0 * ulp[nonzero]), (err / ulp)[nonzero].max()
    assert np.all(got[~nonzero] == 0.0)
    # the reflections round to the double nearest pi/2 and pi
    np.testing.assert_array_equal(angle(1, [0.0, -1.0, 1.0], [1.0, 0.0, 1.0]),
                                  [np.pi / 2, np.pi, np.pi / 4])


def test_asin(fn):
    rng = np.random.default_rng(4)
    x = np.concatenate([rng.uniform(0, 1, 3000), 10.0 ** rng.uniform(-15, 0, 500),
                        1 - 10.0 ** rng.uniform(-16, 0, 500), [0.5, np.nextafter(0.5, 1), 1.0]])
    got = fn(4, x)
    exact = [mpmath.asin(mpmath.mpf(v)) for v in x]
    ulp = np.array([float(abs(mpmath.mpf(g) - e)) for g, e in zip(got, exact)]) / np.spacing(got)
    assert ulp.max() <= 2.0, ulp.max()
    assert fn(4, np.array([0.0]))[0] == 0.0 and fn(4, np.array([1.0]))[0] == np.pi / 2
    assert np.isnan(fn(4, np.array([np.nan]))[0])


def pow_exact(x, p, factor):
    return [mpmath.mpf(factor) * mpmath.mpf(v) ** mpmath.mpf(p) for v in x]


# -delta/2 and -alpha/2 (delta, alpha in [-12, 2]) over squared radii, gamma in [1/2, 6] over g;
# the registry's are -0.233, -0.67 and 0.942
@pytest.mark.parametrize("p", [-0.2334313, -0.67, 0.942, -1.0, -0.5, 0.0, 0.5, 1.0, 2.5, 6.0])
@pytest.mark.parametrize("lo,hi", [(-8.0, 6.0), (-101.0, 155.0)])
def test_power(power, p, lo, hi):
    """Four roundings (two table entries, two products) of at most 2^-53 each, the series'
    (below 0.02) and its first term left out, 8.4e-17 = 0.76 2^-53 times |binom(p, 6)|. The
    mean: four independent errors uniform in +-2^-53 / m have 0.41 each in the root mean
    square, 0.83 together, 0.66 in the mean; the term left out a seventh of its largest."""
    if (hi - lo) * abs(p) > 500:
        lo, hi = -500 / abs(p) / 2, 500 / abs(p) / 2
    rng = np.random.default_rng(int(10 * p) + 50)
    x = 2.0 ** rng.uniform(max(lo, -100.9), min(hi, 154.9), 4000)
    factor = 3.0 * 1.13e-7
    err = relative(power(p, x, factor), pow_exact(x, p, factor))
    left = 0.76 * abs(float(mpmath.binomial(p, 6)))
    assert err.max() <= 4.02 + left, err.max()
    assert err.mean() <= 0.75 + left / 7, err.mean()


def test_power_table_edges(power):
    """Every exponent of the table, at both ends of its mantissas; 2^0 = 1 exactly."""
    e = np.arange(-100, 155)
    x = np.concatenate([2.0**e * 0.5, 2.0 ** e * np.nextafter(1.0, 0)])
    for p in (-0.67, 1.0):
        assert relative(power(p, x), pow_exact(x, p, 1.0)).max() <= 4.1
    e = np.arange(-253, 3)
    x = np.concatenate([2.0 ** (e - 1), 2.0 ** e * np.nextafter(1.0, 0)])
    assert relative(power(0.942, x, 1.0, -253), pow_exact(x, 0.942, 1.0)).max() <= 4.1
    assert power(0.0, np.array([0.3]), 2.5)[0] == 2.5
    assert np.isnan(power(0.5, np.array([np.nan]))[0])


def test_temperature_on_the_table_axis(power):
    """T/dT - T_first/dT + 1: the two factors' roundings (three of 2^-53) of T/dT and one of
    the result; the product itself is not rounded."""
    p, factor, less = -0.2334313, 286.0 / 5.0, 7.0
    x = 2.0 ** np.random.default_rng(8).uniform(-8, 6, 4000)
    got = power(p, x, factor, less=less)
    exact = [v - mpmath.mpf(less) for v in pow_exact(x, p, factor)]
    err = np.array([float(abs(mpmath.mpf(g) - e)) for g, e in zip(got, exact)])
    T = np.array([float(v) for v in pow_exact(x, p, factor)])
    assert np.all(err <= (3.05 * T + np.abs(got)) * EPS)
