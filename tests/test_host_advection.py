"""CPU: advection by the shift with dissipation (advdis of oaxis_rhs.h, interior
form) against the upwinded stencils it rewrites (derivadvect.f90:105-175,
dissipation.f90:181-199), both in double precision and in 80-bit.  In 80-bit the
two are one expression (equal to 1e-17 of the terms' size); in double precision
the rewritten form's error is at most the stencils' own, in the root mean
square over random fields, with and without contraction of products into sums.
Fields that the grid resolves: near one, as the lapse and the metric; near zero,
as the shift and the curvature; steep; and with noise of 1e-3 on them.  (White
noise alone, whose neighbours share no leading bits, is not among them: nothing
cancels there and both forms round at 2^-53 of the value, the rewritten one 1.4
times as much.)"""
import ctypes

import numpy as np
import pytest

import host_probe

PROBE = r"""
#include <random>
#include "oaxis_device.h"
#include "oaxis_rhs.h"
using namespace oax;

struct Patch {
  const double* p;
  double operator()(int i, int j) const { return p[(i - 7) * 7 + (j - 7)]; }   // points 7 .. 13
};

// the stencils in 80-bit: t = 1 for beta <= 0, else mirrored and negated
template <class F>
static long double upwind(const F& f, double beta, int di, int dj, long double q) {
  const int t = beta <= 0.0 ? 1 : -1;
  auto l = [&](int k) { return static_cast<long double>(f(10 + k * t * di, 10 + k * t * dj)); };
  return beta * q * t * (3 * l(1) + 10 * l(0) - 18 * l(-1) + 6 * l(-2) - l(-3));
}
template <class F>
static long double sixth(const F& f) {
  long double s = 40 * static_cast<long double>(f(10, 10));
  const int w[3] = {-15, 6, -1};
  for (int k = 1; k <= 3; ++k)
    s += w[k - 1] * (static_cast<long double>(f(10 + k, 10)) + f(10 - k, 10) + f(10, 10 + k) + f(10, 10 - k));
  return s;
}

// mean squares over n random patches: out[0] of the stencils' error, out[1] of
// advdis's, out[2] of the value
extern "C" void errors(int adv, int dis, double mean, double slope, double noise, int n, double* out) {
  KGrid G{};
  G.Nr = G.Nz = 100; G.g = 3; G.jlo = 1; G.eqsym = 1;
  G.dr = G.dz = 0.1; G.idr = G.idz = 10.0; G.dt = 0.025;
  KPhys P{};
  P.shiftadvect = 1;
  KStencil W{};
  W.r12 = W.z12 = G.idr / 12.0;
  const double up[3] = {10.5, -3.0, 0.5};
  for (int k = 0; k < 3; ++k) W.ar[k] = W.az[k] = up[k] * G.idr / 12.0;
  W.ur = W.uz = 0.5 * G.idr / 12.0;
  const double ds = dis ? 0.1 / G.dt : 0.0, ko = ds * 0.05;
  std::mt19937_64 gen(adv * 2 + dis + 1);
  std::normal_distribution<double> nd;
  for (int k = 0; k < 3; ++k) out[k] = 0.0;
  for (int q = 0; q < n; ++q) {
    double a[6], p[49];
    for (double& v : a) v = slope * nd(gen);
    for (int i = 0; i < 7; ++i)
      for (int j = 0; j < 7; ++j) {
        const double x = 0.1 * (i - 3), y = 0.1 * (j - 3);
        p[i * 7 + j] = mean + a[0] * x + a[1] * y + a[2] * x * x + a[3] * x * y + a[4] * y * y + a[5] * x * x * x +
                       noise * nd(gen);
      }
    const Patch f{p};
    const double br = 0.3 * nd(gen), bz = 0.3 * nd(gen);
    double plain = br * s_adr<true>(f, G, 10, 10, br) + bz * s_adz<true>(f, G, 10, 10, bz);
    if (dis) plain -= s_ko<true>(f, G, 10, 10, ds);
    const double split = adv == 2 ? advdis<true, 2>(f, G, P, W, 10, 10, br, bz, ko, dis != 0)
                                  : advdis<true, 1>(f, G, P, W, 10, 10, br, bz, ko, dis != 0);
    const long double quarter = static_cast<long double>(G.idr) / 12;
    long double exact = upwind(f, br, 1, 0, quarter) + upwind(f, bz, 0, 1, quarter);
    if (dis) exact -= static_cast<long double>(ds) / 20 * sixth(f);
    out[0] += static_cast<double>((plain - exact) * (plain - exact)) / n;
    out[1] += static_cast<double>((split - exact) * (split - exact)) / n;
    out[2] += static_cast<double>(exact * exact) / n;
  }
}
"""

FIELDS = {"near_one": (1.0, 0.1, 0.0), "steep": (1.0, 1.0, 0.0), "near_zero": (0.0, 0.1, 0.0),
          "noisy": (1.0, 0.1, 1e-3)}


@pytest.fixture(scope="module", params=["plain", "contracted"])
def probe(request, tmp_path_factory, oaxis_mod):
    if request.param == "contracted" and " fma " not in open("/proc/cpuinfo").read():
        pytest.skip("this processor has no fused multiply-add")
    flags = ("-O2", "-ffp-contract=off") if request.param == "plain" else ("-O2", "-mfma", "-ffp-contract=fast")
    return host_probe.build(tmp_path_factory.mktemp("adv"), PROBE, flags)


@pytest.mark.parametrize("adv", [1, 2])
@pytest.mark.parametrize("dis", [0, 1])
@pytest.mark.parametrize("field", sorted(FIELDS))
def test_error_is_at_most_that_of_the_stencils(probe, adv, dis, field):
    out = (ctypes.c_double * 3)()
    probe.errors(adv, dis, *(ctypes.c_double(v) for v in FIELDS[field]), 50000, out)
    plain, split, value = (np.sqrt(v) for v in out)
    print("%s adv %d dis %d: stencils %.2e, rewritten %.2e of %.2e" % (field, adv, dis, plain, split, value))
    assert 0.0 < value and plain < 1e-13 * max(value, 1.0)
    assert split <= plain
