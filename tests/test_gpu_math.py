"""The FP64 kernels' own square root and power against correctly rounded values, over the arguments that
the kernels meet and at zero, the ends of the range, infinities, negative arguments and NaN.

Bounds.  Square root: the nearest double (numpy's) for arguments in [1e-290, 1e290], from which the last
residual step rounds once; 4 ulp below, where that step's residual underflows.  Power: 0.75 ulp of the
80-bit result, the last rounding (0.5) and the ends of its two series and two-part sums (each below
2^-4 ulp); where the call goes to the device library (|a ln x| >= 700) 2 ulp."""
import numpy as np
import pytest

import porturb_amd as pa

pytestmark = pytest.mark.gpu

INF, NAN = np.inf, np.nan


def error_in_ulps(y, exact):
    nearest = exact.astype(np.float64)
    return np.abs((y.astype(np.longdouble) - exact) / np.spacing(np.abs(nearest)).astype(np.longdouble)).astype(np.float64)


@pytest.mark.parametrize("lo,hi", [(1e-6, 10.), (1., 4.), (1e-290, 1e290)])
def test_root_is_correctly_rounded(lo, hi):
    x = np.exp(np.random.default_rng(3).uniform(np.log(lo), np.log(hi), 200001))
    assert np.array_equal(pa.eval_fp64("root", x), np.sqrt(x))


def test_root_of_special_arguments():
    x = np.array([0., INF, -1., -1e-310, -INF, NAN, 1.7e308])
    assert np.array_equal(pa.eval_fp64("root", x), [0., INF, NAN, NAN, NAN, NAN, np.sqrt(1.7e308)], equal_nan=True)
    tiny = np.array([5e-324, 1e-310, 2.3e-308, 1e-300])
    assert error_in_ulps(pa.eval_fp64("root", tiny), np.sqrt(tiny.astype(np.longdouble))).max() <= 4.


# rho theta, (p / C0), theta and rho under the exponents of the equation of state and the wall extrapolation
GAMMA = 1003. / 716.


@pytest.mark.parametrize("lo,hi,a", [(200., 400., GAMMA), (1e2, 1e4, 1 / GAMMA), (0.2, 1.5, GAMMA - 1), (0.4, 1.3, 1 / (GAMMA - 1)),
                                     (1e-5, 1e6, -2.5), (1e-300, 1e300, 1 / GAMMA), (1 - 1e-9, 1 + 1e-9, GAMMA)])
def test_power(lo, hi, a):
    x = np.exp(np.random.default_rng(4).uniform(np.log(lo), np.log(hi), 200001))
    assert error_in_ulps(pa.eval_fp64("power", x, a), np.power(x.astype(np.longdouble), np.longdouble(a))).max() <= 0.75


@pytest.mark.parametrize("a", [GAMMA, 1 / GAMMA, GAMMA - 1, -2.5])
def test_power_of_special_arguments(a):
    x = np.array([0., INF, -1., -INF, NAN, 1.])
    with np.errstate(all="ignore"):
        want = np.power(x, a)
    assert np.array_equal(pa.eval_fp64("power", x, a), want, equal_nan=True)
    tiny = np.array([5e-324, 1e-310, 2.3e-308])
    if a > 0:
        exact = np.power(tiny.astype(np.longdouble), np.longdouble(a))
        inside = exact > 3e-308
        assert error_in_ulps(pa.eval_fp64("power", tiny, a), exact)[inside].max(initial=0.) <= 2.


@pytest.mark.parametrize("sign", [1, -1])
def test_power_around_the_hand_over_to_the_library(sign):
    """|a ln x| just below and above 700."""
    x = np.exp(np.linspace(69.9, 70.1, 2001))
    y = pa.eval_fp64("power", x, 10. * sign)
    exact = np.power(x.astype(np.longdouble), np.longdouble(10. * sign))
    err = error_in_ulps(y, exact)
    inside = 10 * np.log(x) < 699.99
    assert err[inside].max() <= 0.75 and err.max() <= 2.
