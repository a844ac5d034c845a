"""CPU: the last substep of a step writes over the step's start y_p
(onestep.f90:129-342 keeps var_p and var apart; the library's three slabs per
level do not), and finebound rides on that launch.  Both are right in place
only under two rules of the per-point code, checked here on a host build of it:

  finebound_point   a group of fields asks for the step's start of the fields
                    that it writes and of no others, the groups' fields are
                    disjoint, and no two records of a zone are one point
  rhs_roles         a part's output does not depend on whether y_p is the
                    output plane, nor on which part ran before it
  rhs_point         likewise for the two-phase form

Outputs are compared bit for bit (one build of one expression)."""
import ctypes

import numpy as np
import pytest

import host_probe

PROBE = r"""
#include <vector>
#include <set>
#include "oaxis_device.h"
#include "oaxis_rhs.h"
using namespace oax;

static KGrid grid(int Nr, int Nz, int eqsym, double h) {
  KGrid G{};
  G.Nr = Nr; G.Nz = Nz; G.g = 3; G.ld = (Nz + 3 + 15) / 16 * 16;
  G.plane = static_cast<long>(Nr + 3) * G.ld;
  G.eqsym = eqsym; G.jlo = eqsym ? 1 : -2;
  G.dr = G.dz = h; G.dt = 0.25 * h; G.idr = G.idz = 1.0 / h;
  G.zoff = eqsym ? 0.5 : 0.5 * (Nz - 3 + 1);
  return G;
}

template <bool SH, bool SC>
static int finebound_rule(int eqsym, int depth, int time0, int chimethod, const double* noise, long n) {
  const KGrid Gf = grid(24, 31, eqsym, 0.1), Gc = grid(24, 31, eqsym, 0.2);
  constexpr int nf = nslots(SH, SC), groups = finebound_groups(SH, SC);
  KPhys P{};
  P.chimethod = chimethod;
  KTime T{};
  T.border = 2; T.depth = depth; T.same = 0;
  T.c0 = 0.5; T.c1 = 0.75; T.c2 = -0.25;
  std::vector<double> yc(nf * Gc.plane), strip(nf * 3 * 64);
  for (size_t q = 0; q < yc.size(); ++q) yc[q] = 1.0 + 0.01 * noise[q % n];
  for (size_t q = 0; q < strip.size(); ++q) strip[q] = 1.0 + 0.01 * noise[(7 * q) % n];
  std::set<long> points;
  for (long q = 0; q < fb_count(Gf, depth); ++q) {
    FbPoint fp{};
    fb_geometry(Gf, Gc, depth, 1, q, fp);
    if (fp.which < 0) continue;
    if (!points.insert(IDX(Gf, fp.i, fp.j)).second) return 1;      // a point with two records
    unsigned all = 0;
    for (int grp = 0; grp < groups; ++grp) {
      std::vector<double> yf(nf * Gf.plane, -7.0);
      unsigned read = 0, wrote = 0;
      finebound_point<SH, SC>(Gf, Gc, P, T, time0, yc.data(), yf.data(), strip.data(), strip.data(), strip.data(), fp,
                              grp, [&](int s) { read |= 1u << s; return 1.0; });
      for (int s = 0; s < nf; ++s) {
        if (yf[s * Gf.plane + IDX(Gf, fp.i, fp.j)] != -7.0) wrote |= 1u << s;
        for (long k = 0; k < Gf.plane; ++k) {
          if (yf[s * Gf.plane + k] == -7.0) continue;
          const int i = static_cast<int>(k / Gf.ld) - 2, j = static_cast<int>(k % Gf.ld) - 2;
          const int im = i < 1 ? 1 - i : i, jm = (eqsym && j < 1) ? 1 - j : j;
          if (im != fp.i || jm != fp.j) return 2;                  // neither the point nor an image
        }
      }
      if (read & ~wrote) return 3;                                 // asks for a field of another group
      if (wrote & all) return 4;                                   // two groups write one field
      all |= wrote;
    }
  }
  return 0;
}

extern "C" int check_finebound(int sh, int sc, int eqsym, int depth, int time0, int chimethod, const double* noise,
                               long n) {
  if (sh && sc) return finebound_rule<true, true>(eqsym, depth, time0, chimethod, noise, n);
  if (sh) return finebound_rule<true, false>(eqsym, depth, time0, chimethod, noise, n);
  if (sc) return finebound_rule<false, true>(eqsym, depth, time0, chimethod, noise, n);
  return finebound_rule<false, false>(eqsym, depth, time0, chimethod, noise, n);
}

struct Setup {
  KGrid G; KPhys P; KStep S; KStencil W;
};

static Setup setup(int eqsym, int rk4, int time0, int chimethod) {
  Setup u{};
  u.G = grid(20, 23, eqsym, 0.1);
  u.P.slicing = OA_SLICING_1PLUSLOG; u.P.gauge_f = 2.0; u.P.geodiss = 0.1; u.P.scalardiss = 0.1; u.P.eta = 2.0;
  u.P.drivercsi = 0.75; u.P.drivereta = 0.5; u.P.driveradv = 1; u.P.shiftadvect = 1;
  u.P.scalarmethod = OA_SCALARMETHOD_FIRST; u.P.chimethod = chimethod; u.P.radiative = 1;
  const int n = rk4 ? 4 : 3;
  u.S = KStep{n, n, rk4, u.G.dt, rk4 ? 1.0 / 6 : 0.0, time0, nullptr};
  const KGrid& G = u.G;
  u.W.r12 = u.W.z12 = G.idr / 12.0; u.W.rr12 = u.W.zz12 = G.idr * G.idr / 12.0;
  u.W.rz3 = G.idr * G.idz / 3.0; u.W.rz48 = G.idr * G.idz / 48.0;
  const double up[3] = {10.5, -3.0, 0.5};
  for (int k = 0; k < 3; ++k) u.W.ar[k] = u.W.az[k] = up[k] * G.idr / 12.0;
  u.W.ur = u.W.uz = 0.5 * G.idr / 12.0;
  u.W.ko_g = u.W.ko_s = 0.1 / G.dt * 0.05;
  return u;
}

static void fill(std::vector<double>& y, const KGrid& G, int nf, const double* noise, long n, int shift) {
  for (int s = 0; s < nf; ++s)
    for (long k = 0; k < G.plane; ++k) {
      const bool one = s == S_alpha || s == S_chi || s == S_A || s == S_B || s == S_H;
      y[s * G.plane + k] = (one ? 1.0 : 0.0) + 0.01 * noise[(s * 131 + k * shift) % n];
    }
}

template <bool SH, bool SC, int ROLE>
static void run_role(const Setup& u, const std::vector<double>& yin, const double* yp, std::vector<double>& acc,
                     double* yout) {
  const KGrid& G = u.G;
  for (int i = 1; i <= G.Nr; ++i) {
    double ri[5];
    for (int q = 0; q < 5; ++q) ri[q] = 1.0 / ((i + q - 2 - 0.5) * G.dr);
    const RoleView V{yin.data(), 1 - G.g, 1 - G.g, G.ld, static_cast<int>(G.plane), ri + 2,
                     SH ? shift_slot(SH_dtbeta_r) : 0, 0};
    for (int j = G.jlo; j <= G.Nz; ++j)
      rhs_roles<SH, SC, false, false, ROLE>(G, u.P, u.S, u.W, V, yp, acc.data(), yout, i, j);
  }
}

template <bool SH, bool SC>
static int roles_rule(int eqsym, int rk4, int time0, int chimethod, const double* noise, long n) {
  const Setup u = setup(eqsym, rk4, time0, chimethod);
  constexpr int nf = nslots(SH, SC);
  constexpr int R0 = ROLE_K | (SH && SC ? ROLE_SCALAR : ROLE_LAPSE);
  constexpr int R1 = (ROLE_DELTA | ROLE_LAPSE | ROLE_METRIC | ROLE_SCALAR) & ~R0;
  const size_t size = nf * u.G.plane;
  std::vector<double> yin(size), yp(size), acc(size), apart;
  fill(yin, u.G, nf, noise, n, 1);
  fill(yp, u.G, nf, noise, n, 3);
  fill(acc, u.G, nf, noise, n, 5);
  apart = yp;                          // what a substep leaves alone is alike on both sides
  std::vector<double> a = acc;
  run_role<SH, SC, R0>(u, yin, yp.data(), a, apart.data());
  run_role<SH, SC, R1>(u, yin, yp.data(), a, apart.data());
  for (int order = 0; order < 2; ++order) {
    std::vector<double> y = yp, b = acc;
    if (order == 0) run_role<SH, SC, R0>(u, yin, y.data(), b, y.data());
    run_role<SH, SC, R1>(u, yin, y.data(), b, y.data());
    if (order == 1) run_role<SH, SC, R0>(u, yin, y.data(), b, y.data());
    for (size_t q = 0; q < size; ++q)
      if (!(y[q] == apart[q]) && !(y[q] != y[q] && apart[q] != apart[q])) return 1 + order;
  }
  if (apart == yp) return 3;           // nothing was advanced
  return 0;
}

extern "C" int check_roles(int sh, int sc, int eqsym, int rk4, int time0, int chimethod, const double* noise, long n) {
  if (sh && sc) return roles_rule<true, true>(eqsym, rk4, time0, chimethod, noise, n);
  if (sc) return roles_rule<false, true>(eqsym, rk4, time0, chimethod, noise, n);
  return roles_rule<false, false>(eqsym, rk4, time0, chimethod, noise, n);
}

extern "C" int check_phases(int eqsym, int rk4, int time0, int chimethod, const double* noise, long n) {
  const Setup u = setup(eqsym, rk4, time0, chimethod);
  const KGrid& G = u.G;
  constexpr int nf = nslots(true, false);
  const size_t size = nf * G.plane;
  std::vector<double> yin(size), yp(size), acc(size), gaux(NAUX * G.plane), apart, y;
  fill(yin, G, nf, noise, n, 1);
  fill(yp, G, nf, noise, n, 3);
  fill(acc, G, nf, noise, n, 5);
  apart = yp;
  y = yp;
  const TileView V{yin.data(), 1 - G.g, 1 - G.g, G.ld, static_cast<int>(G.plane), nf};
  for (int i = 1; i <= G.Nr; ++i)
    for (int j = G.jlo; j <= G.Nz; ++j) {
      rhs_point<false, false, false, 1>(G, u.P, u.S, V, nullptr, nullptr, nullptr, gaux.data(), i, j);
      rhs_point<true, false, false, 2>(G, u.P, u.S, V, yp.data(), acc.data(), apart.data(), gaux.data(), i, j);
      rhs_point<true, false, false, 2>(G, u.P, u.S, V, y.data(), acc.data(), y.data(), gaux.data(), i, j);
    }
  for (size_t q = 0; q < size; ++q)
    if (!(y[q] == apart[q]) && !(y[q] != y[q] && apart[q] != apart[q])) return 1;
  return apart == yp ? 3 : 0;
}
"""

N = 100003          # prime, so that the planes' strides through it differ


@pytest.fixture(scope="module")
def probe(tmp_path_factory, oaxis_mod):
    lib = host_probe.build(tmp_path_factory.mktemp("in_place"), PROBE)
    noise = np.random.default_rng(5).standard_normal(N)
    return lib, noise.ctypes.data_as(ctypes.POINTER(ctypes.c_double)), noise


@pytest.mark.parametrize("shift,scalar", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("depth", [2, 5])
def test_finebound_groups_read_what_they_write(probe, shift, scalar, depth):
    lib, p, _ = probe
    for eqsym in (0, 1):
        for time0 in (0, 1):
            for chimethod in (0, 1):
                rc = lib.check_finebound(shift, scalar, eqsym, depth, time0, chimethod, p, ctypes.c_long(N))
                assert rc == 0, (rc, eqsym, time0, chimethod)


@pytest.mark.parametrize("shift,scalar", [(0, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("eqsym", [0, 1])
def test_parts_advance_a_level_in_place(probe, shift, scalar, eqsym):
    lib, p, _ = probe
    for rk4 in (0, 1):
        for time0 in (0, 1):
            for chimethod in (0, 1):
                rc = lib.check_roles(shift, scalar, eqsym, rk4, time0, chimethod, p, ctypes.c_long(N))
                assert rc == 0, (rc, rk4, time0, chimethod)


@pytest.mark.parametrize("eqsym", [0, 1])
def test_two_phases_advance_a_level_in_place(probe, eqsym):
    lib, p, _ = probe
    for rk4 in (0, 1):
        for time0 in (0, 1):
            for chimethod in (0, 1):
                rc = lib.check_phases(eqsym, rk4, time0, chimethod, p, ctypes.c_long(N))
                assert rc == 0, (rc, rk4, time0, chimethod)
