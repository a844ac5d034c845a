"""CPU: the horizon finder's shared reciprocals (oaxis_recip.h) against
division, on a host build whose first estimate has the hardware's accuracy
(2^-24) and is off by as much to either side.

Bounds, from the two Newton steps: the reciprocal before its last rounding is
off by 2^-96 of itself, so it is the correctly rounded one for every divisor
whose reciprocal is not that close to the middle of two numbers, and the
quotient is then that of a division (Markstein 1990).  A random divisor misses
with a chance of about 2^-40.  By 2 - 2^-52, whose reciprocal is 2^-106 from
a middle, a quotient may be one unit in the last place off and no more."""
import ctypes

import numpy as np
import pytest

import host_probe

PROBE = r"""
#include <cmath>
static double estimate_error = 0.0;
// a reciprocal good to 2^-24, whatever the exponent
static double estimate(double d) {
  int e;
  const double m = std::frexp(d, &e);
  const double f = static_cast<double>(1.0f / static_cast<float>(m)) * (1.0 + estimate_error);
  return std::ldexp(f, -e);
}
#define OA_RCP(d) estimate(d)
#define OA_HD inline
using std::fma;
#include "oaxis_recip.h"
extern "C" void set_error(double e) { estimate_error = e; }
extern "C" void quotients(long n, const double* x, const double* d, double* out) {
  for (long q = 0; q < n; ++q) out[q] = oax::AhRecip(d[q]).of(x[q]);
}
extern "C" void over(long n, const double* x, const int* m, double* out) {
  for (long q = 0; q < n; ++q) out[q] = oax::ah_over(x[q], m[q]);
}
"""

DP = ctypes.POINTER(ctypes.c_double)


@pytest.fixture(scope="module")
def probe(tmp_path_factory, oaxis_mod):
    return host_probe.build(tmp_path_factory.mktemp("recip"), PROBE)


def quotients(lib, x, d, error):
    lib.set_error(ctypes.c_double(error))
    out = np.empty_like(x)
    lib.quotients(ctypes.c_long(x.size), x.ctypes.data_as(DP), d.ctypes.data_as(DP), out.ctypes.data_as(DP))
    return out


def numbers(rng, n, lo, hi):
    """Normal numbers of both signs with exponents spread over [lo, hi]."""
    return np.ldexp(rng.uniform(1.0, 2.0, n), rng.integers(lo, hi, n)) * rng.choice((-1.0, 1.0), n)


@pytest.mark.parametrize("error", [0.0, 2.0 ** -24, -2.0 ** -24])
@pytest.mark.parametrize("spread", [1, 300])
def test_quotients_are_those_of_division(probe, error, spread):
    rng = np.random.default_rng(7)
    n = 1 << 20
    x, d = numbers(rng, n, -spread, spread + 1), numbers(rng, n, -spread, spread + 1)
    got = quotients(probe, x, d, error)
    assert np.array_equal(got, x / d)
    # exact quotients, and zeros
    k = np.ldexp(rng.integers(1, 1 << 26, n).astype(float), -8)
    d = rng.integers(1, 1 << 26, n).astype(float)
    assert np.array_equal(quotients(probe, k * d, d, error), k)
    assert np.array_equal(quotients(probe, np.zeros(n), d, error), np.zeros(n))


@pytest.mark.parametrize("error", [0.0, 2.0 ** -24, -2.0 ** -24])
def test_divisors_next_to_a_middle_are_one_unit_off_at_most(probe, error):
    rng = np.random.default_rng(8)
    d = np.ldexp(np.full(1 << 16, 2.0 - 2.0 ** -52), rng.integers(-20, 20, 1 << 16))
    x = numbers(rng, d.size, -20, 20)
    x[:64] = np.ldexp(1.0, np.arange(64) - 32)
    got, want = quotients(probe, x, d, error), x / d
    assert np.all(np.abs(got - want) <= np.spacing(np.abs(want)))


def test_weights_divide_by_small_integers(probe):
    rng = np.random.default_rng(9)
    x = numbers(rng, 1 << 18, -60, 60)
    m = rng.choice(np.array([-3, -2, -1, 1, 2, 3], dtype=np.int32), x.size)
    out = np.empty_like(x)
    probe.over(ctypes.c_long(x.size), x.ctypes.data_as(DP), m.ctypes.data_as(ctypes.POINTER(ctypes.c_int)),
               out.ctypes.data_as(DP))
    assert np.array_equal(out, x / m)
