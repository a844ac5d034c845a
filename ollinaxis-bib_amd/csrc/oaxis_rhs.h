// The right-hand side split by parts: which waves form which sources of a
// point, and every source with its RK update.  Included by oaxis_kernels.hip
// after oaxis_device.h, whose stencils and phi-mode rules (rhs_point) it
// shares.
#pragma once

#include "oaxis_device.h"

namespace oax {

// The staged tile as rhs_roles reads it.  dtb(k, pre) is the plane dtbeta_r
// (k = 0) or dtbeta_z is differentiated from: with pre, that of the dtbeta
// state that the first substep after the initial auxiliary pass
// differentiates (KStep::dtb_pre), staged after the evolved fields.  inv_r(k)
// is 1 / r of the column i + k, |k| <= 2, from the block's table.
struct RoleView {
  const double* t;      // slot 0's value of point (ib, jb)
  int ib, jb, tw, ts;
  const double* ri;     // 1 / r of this point's column
  int ndtb, npre;       // tile slots of dtbeta_r and of its first-substep form
  OA_HD TilePlane fld(int s) const { return TilePlane{t + s * ts, ib, jb, tw}; }
  OA_HD TilePlane dtb(int k, bool pre) const { return fld((pre ? npre : ndtb) + k); }
  OA_HD double inv_r(int k) const { return ri[k]; }
};

// gradient and second derivatives with the folded weights where every
// stencil is centred (IN), the reference's closures elsewhere
template <bool IN, class F>
OA_HD D1 grad(const F& f, const KGrid& G, const KStencil& W, int i, int j) {
  if constexpr (IN)
    return {W.r12 * (8.0 * (f(i + 1, j) - f(i - 1, j)) - (f(i + 2, j) - f(i - 2, j))),
            W.z12 * (8.0 * (f(i, j + 1) - f(i, j - 1)) - (f(i, j + 2) - f(i, j - 2)))};
  else
    return {s_d1r(f, G, i, j), s_d1z(f, G, i, j)};
}
// one component of it: DIR = 0 along r, 1 along z
template <bool IN, int DIR, class F>
OA_HD double s_d1(const F& f, const KGrid& G, const KStencil& W, int i, int j) {
  if constexpr (IN && DIR == 0) return W.r12 * (8.0 * (f(i + 1, j) - f(i - 1, j)) - (f(i + 2, j) - f(i - 2, j)));
  else if constexpr (IN) return W.z12 * (8.0 * (f(i, j + 1) - f(i, j - 1)) - (f(i, j + 2) - f(i, j - 2)));
  else if constexpr (DIR == 0) return s_d1r(f, G, i, j);
  else return s_d1z(f, G, i, j);
}
// The differences are summed in the order of s_d2r, s_d2z and s_d2rz: it is
// their rounding, of order one ulp of f over h^2, that the sources see.
template <bool IN, class F>
OA_HD D2 hess(const F& f, const KGrid& G, const KStencil& W, int i, int j) {
  if constexpr (IN) {
    const double c = f(i, j);
    const double rp = f(i + 1, j), rm = f(i - 1, j), rp2 = f(i + 2, j), rm2 = f(i - 2, j);
    const double zp = f(i, j + 1), zm = f(i, j - 1), zp2 = f(i, j + 2), zm2 = f(i, j - 2);
    D2 d;
    d.r = W.r12 * (8.0 * (rp - rm) - (rp2 - rm2));
    d.z = W.z12 * (8.0 * (zp - zm) - (zp2 - zm2));
    d.rr = -W.rr12 * (30.0 * c - 16.0 * (rp + rm) + rp2 + rm2);
    d.zz = -W.zz12 * (30.0 * c - 16.0 * (zp + zm) + zp2 + zm2);
    d.rz = W.rz3 * (f(i + 1, j + 1) + f(i - 1, j - 1) - f(i + 1, j - 1) - f(i - 1, j + 1))
           - W.rz48 * (f(i + 2, j + 2) + f(i - 2, j - 2) - f(i + 2, j - 2) - f(i - 2, j + 2));
    return d;
  } else {
    return {s_d1r(f, G, i, j), s_d1z(f, G, i, j), s_d2r(f, G, i, j), s_d2z(f, G, i, j), s_d2rz(f, G, i, j)};
  }
}

// Advection by the shift and Kreiss-Oliger dissipation of one field:
//   br adv_r f + bz adv_z f - ko D6 f          (ADV: with the first two terms)
// The upwinded derivative (derivadvect.f90:105-175) is q (3 f1 + 10 f0 -
// 18 f-1 + 6 f-2 - f-3) for beta <= 0 and minus its mirror image for beta >
// 0.  Its odd part is q/2 (21 (f1 - f-1) - 6 (f2 - f-2) + (f3 - f-3)); its
// even part is -sign(beta) q/2 times the sixth difference D6 that the
// dissipation needs anyway, so beta times it is -|beta| q/2 D6: both upwind
// sides cost one expression, without a branch or a select.  With centred
// advection (shiftadvect = .false.) the weights are those of the centred
// derivative; the scalar field is upwinded always (ADV = 2).
//
// The weights of this sum are larger than the upwind stencil's (60/12 of f/h
// against 38/12), and summed over the values f themselves it rounds up to 1.6
// times as far off.  So it is summed over the differences f(k) - f(0), which
// are exact, or nearly so, wherever the grid resolves f: the error is then 0.01
// to 0.25 of the stencil's on fields near one and 0.7 to 0.9 of it on fields near
// zero.  The differences replace the values in registers; the 12 additions more
// cost a batch of 16 pulses 69.5 -> 70.6 ms, less than its runs differ by.
template <bool IN, int ADV, class F>
OA_HD double advdis(const F& f, const KGrid& G, const KPhys& P, const KStencil& W, int i, int j, double br, double bz,
                    double ko, bool dis) {
  if constexpr (IN) {
    const double c = f(i, j);
    const double rp = f(i + 1, j), rm = f(i - 1, j), rp2 = f(i + 2, j), rm2 = f(i - 2, j);
    const double rp3 = f(i + 3, j), rm3 = f(i - 3, j);
    const double zp = f(i, j + 1), zm = f(i, j - 1), zp2 = f(i, j + 2), zm2 = f(i, j - 2);
    const double zp3 = f(i, j + 3), zm3 = f(i, j - 3);
    if constexpr (ADV == 0) {
      const double d6r = 20.0 * c - 15.0 * (rp + rm) + 6.0 * (rp2 + rm2) - (rp3 + rm3);
      const double d6z = 20.0 * c - 15.0 * (zp + zm) + 6.0 * (zp2 + zm2) - (zp3 + zm3);
      return -ko * (d6r + d6z);
    }
    const double ap = rp - c, am = rm - c, ap2 = rp2 - c, am2 = rm2 - c, ap3 = rp3 - c, am3 = rm3 - c;
    const double bp = zp - c, bm = zm - c, bp2 = zp2 - c, bm2 = zm2 - c, bp3 = zp3 - c, bm3 = zm3 - c;
    const double d6r = 6.0 * (ap2 + am2) - 15.0 * (ap + am) - (ap3 + am3);
    const double d6z = 6.0 * (bp2 + bm2) - 15.0 * (bp + bm) - (bp3 + bm3);
    if constexpr (ADV == 2) {
      const double odr = W.r12 * (10.5 * (ap - am) - 3.0 * (ap2 - am2) + 0.5 * (ap3 - am3));
      const double odz = W.z12 * (10.5 * (bp - bm) - 3.0 * (bp2 - bm2) + 0.5 * (bp3 - bm3));
      return br * odr + bz * odz - (ko + 0.5 * W.r12 * fabs(br)) * d6r - (ko + 0.5 * W.z12 * fabs(bz)) * d6z;
    } else {
      const double odr = W.ar[0] * (ap - am) + W.ar[1] * (ap2 - am2) + W.ar[2] * (ap3 - am3);
      const double odz = W.az[0] * (bp - bm) + W.az[1] * (bp2 - bm2) + W.az[2] * (bp3 - bm3);
      return br * odr + bz * odz - (ko + W.ur * fabs(br)) * d6r - (ko + W.uz * fabs(bz)) * d6z;
    }
  } else {
    double s = 0.0;
    if constexpr (ADV != 0) {
      if (ADV == 2 || P.shiftadvect) s = br * s_adr(f, G, i, j, br) + bz * s_adz(f, G, i, j, bz);
      else s = br * s_d1r(f, G, i, j) + bz * s_d1z(f, G, i, j);
    }
    if (dis) s -= s_ko(f, G, i, j, 20.0 * ko);
    return s;
  }
}

// The sources fall into five parts with few intermediate results in common,
// so different waves form them for the same points (ROLE, a bit mask): the
// extrinsic curvature (the Ricci tensor, D_i D_j alpha, K_ij K^ij, matter);
// Delta and the shift (the divergences of KT, the second derivatives of the
// shift); the lapse and the conformal metric, which the projection couples;
// and the scalar field.  Each call forms the sources of its own fields, their
// dissipation, radiative boundaries, RK update and parity images; what a part
// does not use compiles out.
enum RhsRole { ROLE_K = 1, ROLE_DELTA = 2, ROLE_LAPSE = 4, ROLE_METRIC = 8, ROLE_SCALAR = 16 };

// accumulate (prl/arrays.pl:533-599) and update (:1282-1328) of the N slots
// one part owns; y_p and the accumulators of all of them are loaded together
// before the first store (one memory round trip; stores would serialise them).
// On a step's last substep the output plane is y_p itself: a part reads y_p of
// the slots it owns and of no others, at its own point, so the parts of other
// waves may write theirs in any order.
template <int N>
struct RkUpdate {
  double yv[N], av[N];
  bool first, last, rk4;
  double w, dtw;
  double* acc;
  OA_HD RkUpdate(const KStep& S, const double* yp, double* a, const int (&slot)[N], long pl, long k)
      : first(S.iter == 1), last(S.iter == S.niter), rk4(S.rk4 != 0), w(S.w), dtw(S.dtw), acc(a) {
#pragma unroll
    for (int q = 0; q < N; ++q) yv[q] = yp[slot[q] * pl + k];
    if (rk4 && !first) {
#pragma unroll
      for (int q = 0; q < N; ++q) av[q] = a[slot[q] * pl + k];
    } else {
#pragma unroll
      for (int q = 0; q < N; ++q) av[q] = 0.0;
    }
  }
  // slot q's new value from its source
  OA_HD double operator()(int q, long at, double s) const {
    double sv = s;
    if (rk4) {
      const double t = av[q] + w * s;      // av = 0 on the first iteration
      if (last) sv = t;
      else acc[at] = t;
    }
    return yv[q] + dtw * sv;
  }
};

// -D'_m g^im of the conformal metric (auxiliary_geometry.f90:1085-1175),
// differentiated as the products g^ab, like the reference
template <bool IN, class View>
OA_HD void deldef(const View& V, const KGrid& G, const KStencil& W, int i, int j, double r, double gC, double g_lambda,
                  double& Dr_, double& Dz_) {
  const auto FA = V.fld(S_A), FB = V.fld(S_B), FH = V.fld(S_H), FC = V.fld(S_C);
  auto fgA = [&](int ii, int jj) { return FB(ii, jj) * FH(ii, jj); };
  auto fgB = [&](int ii, int jj) { return FA(ii, jj) * FH(ii, jj); };
  auto fgC = [&](int ii, int jj) { return -FC(ii, jj) * FH(ii, jj); };
  const D1 dgC = grad<IN>(fgC, G, W, i, j);
  const double dgA_r = s_d1<IN, 0>(fgA, G, W, i, j), dgB_z = s_d1<IN, 1>(fgB, G, W, i, j);
  Dr_ = -dgA_r - r * dgC.z - r * g_lambda;
  Dz_ = -dgC.r * r - dgB_z - 2.0 * gC;
}

// The connection.  With the flat derivative D' of cylindrical coordinates and
// T_cab = D'_c g_ab of the conformal metric (g_rr = A, g_zz = B, g_rz = r C,
// g_phiphi = r^2 H), the difference of the connections is X_abc = (T_bac +
// T_cab - T_abc) / 2: P_bc = X_rbc and Q_bc = X_zbc in the rho-z block; U, V:
// their first index raised.  The Ricci tensor, div KT and D_i D_j f are
// contractions of these; expanded in the components of the metric, as
// calc_conformalRicci1-4.f90, calc_DIVKTA.f90 and auxiliary_geometry.f90:
// 1268-1324 have them, the same sums take several times the operations.
struct Connection {
  double Prr, Prz, Pzz, Qrr, Qrz, Qzz;
  double Urr, Urz, Uzz, Vrr, Vrz, Vzz;
};

// D_phi D_phi f / r^2 of a scalar (:1268-1324)
OA_HD double hess_H(double fr, double fz, const D1& dH, double r, double ir, double H, double gA, double gB, double gC) {
  return (0.5 * fr * gC * dH.z + 0.5 * fz * gC * dH.r) * r + 0.5 * fr * gA * dH.r + fz * gC * H +
         0.5 * fz * gB * dH.z + fr * gA * H * ir;
}

// derivatives of phi from the state: of phi itself in phi mode, else of chi
template <bool PHIMODE, bool IN, class View>
OA_HD D1 grad_phi(const View& V, const KGrid& G, const KStencil& W, int i, int j, double ic) {
  if constexpr (PHIMODE) return grad<IN>(V.fld(S_phi), G, W, i, j);
  const D1 dc = grad<IN>(V.fld(S_chi), G, W, i, j);
  return {-0.5 * (dc.r * ic), -0.5 * (dc.z * ic)};
}

// matter terms of the real scalar field (auxiliary_matter / stressenergy)
struct Matter {
  double rho, J_r, J_z, S_A, S_B, S_C, trS;
};

template <bool SHIFT, class View>
OA_HD Matter matter_point(const KPhys& P, const View& V, int i, int j, double r, double ir, double A, double B,
                          double H, double C, double gA, double gB, double gH, double gC, double ipsi4, double psi4) {
  Matter m;
  const double xr = V.fld(scalar_slot(SHIFT, SC_xi_r))(i, j), xz = V.fld(scalar_slot(SHIFT, SC_xi_z))(i, j);
  const double pi = V.fld(scalar_slot(SHIFT, SC_pi))(i, j);
  double Vpot = 0.0;
  if (P.scalarpotential != OA_POT_NONE) {
    const double ph = V.fld(scalar_slot(SHIFT, SC_phi))(i, j);
    Vpot = 0.5 * P.scalar_mass * P.scalar_mass * ph * ph;
    if (P.scalarpotential == OA_POT_PHI4) Vpot += 0.25 * P.scalar_lambda * ph * ph * ph * ph;
  }
  const double q2 = (gA * xr * xr + gB * xz * xz + 2.0 * r * gC * xr * xz) * ipsi4;
  m.rho = 0.5 * (pi * pi + q2) + Vpot;
  m.J_r = -(gA * xr + r * gC * xz) * pi * ipsi4;
  m.J_z = -(gB * xz + r * gC * xr) * pi * ipsi4;
  const double aux = 0.5 * (pi * pi - q2) - Vpot;
  m.S_A = xr * xr + A * psi4 * aux;
  m.S_B = xz * xz + B * psi4 * aux;
  m.S_C = xr * xz * ir + C * psi4 * aux;
  const double S_H = H * psi4 * aux;
  m.trS = (gA * m.S_A + gB * m.S_B + gH * S_H + 2.0 * r * r * gC * m.S_C) * ipsi4;
  return m;
}

template <bool SHIFT, bool SCALAR, bool PHIMODE, bool IN, int ROLE, class View>
OA_HD void rhs_roles(const KGrid& G, const KPhys& P, const KStep& S, const KStencil& W, const View& V,
                     const double* yp, double* __restrict__ acc, double* yout, int i, int j) {

  const long pl = G.plane;
  auto fld = [&](int s) { return V.fld(s); };
  const long k = IDX(G, i, j);

  // coordinates (evolve.f90:52-71)
  const double r = (static_cast<double>(i) - 0.5) * G.dr;
  const double z = (static_cast<double>(j) - G.zoff) * G.dz;
  const double ir = V.inv_r(0);
  const double r2 = r * r;

  const auto Fa = fld(S_alpha), Fchi = fld(S_chi), Fphi = fld(S_phi);
  const auto FA = fld(S_A), FB = fld(S_B), FH = fld(S_H), FC = fld(S_C);
  const auto FK = fld(S_trK), FKA = fld(S_KTA), FKB = fld(S_KTB), FKC = fld(S_KTC);
  const auto FDr = fld(S_Delta_r), FDz = fld(S_Delta_z);

  // metric, inverse, conformal factor (:178-236, :325-507); hdet = 1
  const double alpha = Fa(i, j), chi = Fchi(i, j);
  const double A = FA(i, j), B = FB(i, j), H = FH(i, j), C = FC(i, j);
  const double gA = B * H, gB = A * H, gH = 1.0 / H, gC = -C * H;
  const double rgC = r * gC, gH2 = gH * gH;
  const double ipsi4 = chi * chi, ic = 1.0 / chi;
  const double lambda = (A - H) * ir * ir;
  const double g_lambda = C * C - B * lambda;
  const double t23 = 2.0 * third;
  constexpr double smallpi = 3.14159265358979323846;

  double br = 0.0, bz = 0.0;
  if constexpr (SHIFT) {
    br = fld(shift_slot(SH_beta_r))(i, j);
    bz = fld(shift_slot(SH_beta_z))(i, j);
  }
  // advection by the shift, with or without dissipation
  const bool gdis = P.geodiss != 0.0, sdis = P.scalardiss != 0.0;
  auto adv = [&](const auto& f) { return advdis<IN, 1>(f, G, P, W, i, j, br, bz, 0.0, false); };
  auto advko = [&](const auto& f) { return advdis<IN, SHIFT ? 1 : 0>(f, G, P, W, i, j, br, bz, W.ko_g, gdis); };
  auto advkos = [&](const auto& f) { return advdis<IN, SHIFT ? 2 : 0>(f, G, P, W, i, j, br, bz, W.ko_s, sdis); };
  const bool onr = (i == G.Nr), onzR = (j == G.Nz), onzL = (!G.eqsym && j == 1 - G.g);
  const bool bnd = !IN && (onr || onzR || onzL);
  const bool radiative = bnd && P.radiative;

  const bool pt0 = (S.proj_t0 != 0);
  double* const yo = yout;

  // ---- the extrinsic curvature (sources_geometry.f90:77-575)
  if constexpr ((ROLE & ROLE_K) != 0) {
    // the Ricci tensor (:1397-1493, calc_conformalRicci1..4), field by field
    double RA, RB, RC, RH;
    double Dd_r, Dd_z;
    deldef<IN>(V, G, W, i, j, r, gC, g_lambda, Dd_r, Dd_z);
    part(Dd_r, Dd_z);
    {
      // term 2: the derivatives of the evolved Delta
      const double Delta_r = FDr(i, j);
      const D1 dDr = grad<IN>(FDr, G, W, i, j);
      const D1 dDz = grad<IN>(FDz, G, W, i, j);
      RA = C * dDz.r * r + A * dDr.r;
      RB = C * dDr.z * r + B * dDz.z;
      RH = Delta_r * H * ir;
      RC = 0.5 * C * (dDr.r + dDz.z) + 0.5 * (C * Delta_r + A * dDr.z + B * dDz.r) * ir;
    }
    part(RA, RB, RC, RH);
    // term 1: second derivatives of the conformal metric, and the rest of
    // term 2, DelDef^k X_(ij)k
    D1 dA, dB, dH, dC;
    {
      const D2 d = hess<IN>(FA, G, W, i, j);
      dA = D1{d.r, d.z};
      RA += -rgC * d.rz - 0.5 * gB * d.zz - 0.5 * gA * d.rr - 0.5 * gH * d.r * ir + gH * lambda;
      RA += 0.5 * (Dd_r * d.r + Dd_z * d.z);
    }
    part(RA, dA.r, dA.z);
    {
      const D2 d = hess<IN>(FB, G, W, i, j);
      dB = D1{d.r, d.z};
      RB += -rgC * d.rz - 0.5 * gA * d.rr - 0.5 * gB * d.zz - 0.5 * gH * d.r * ir;
      RB += 0.5 * (Dd_r * d.r + Dd_z * d.z);
    }
    part(RB, dB.r, dB.z);
    {
      const D2 d = hess<IN>(FH, G, W, i, j);
      dH = D1{d.r, d.z};
      RH += -rgC * d.rz - 0.5 * gB * d.zz - 0.5 * gA * d.rr - 0.5 * gH * d.r * ir - gH * lambda;
      RH += 0.5 * (Dd_r * d.r + Dd_z * d.z);
    }
    part(RH, dH.r, dH.z);
    {
      const D2 d = hess<IN>(FC, G, W, i, j);
      dC = D1{d.r, d.z};
      RC += -rgC * d.rz - 0.5 * gA * d.rr - gC * d.z - 0.5 * gB * d.zz + (-gA * d.r - 0.5 * gH * d.r) * ir;
      RC += 0.5 * (Dd_r * d.r + Dd_z * d.z);
    }
    part(RC, dC.r, dC.z);
    Connection X;
    {
      const double Trz_r = C + r * dC.r, Trz_z = r * dC.z;
      X.Prr = 0.5 * dA.r; X.Prz = 0.5 * dA.z; X.Pzz = Trz_z - 0.5 * dB.r;
      X.Qrr = Trz_r - 0.5 * dA.z; X.Qrz = 0.5 * dB.r; X.Qzz = 0.5 * dB.z;
      X.Urr = gA * X.Prr + rgC * X.Qrr; X.Urz = gA * X.Prz + rgC * X.Qrz; X.Uzz = gA * X.Pzz + rgC * X.Qzz;
      X.Vrr = rgC * X.Prr + gB * X.Qrr; X.Vrz = rgC * X.Prz + gB * X.Qrz; X.Vzz = rgC * X.Pzz + gB * X.Qzz;
    }
    {
      // terms 3 and 4, quadratic in the connection: g^mn (X^k_mi X_jkn +
      // X^k_mj X_ikn + X^k_im X_kjn), with F_a = X_aphiphi / r^2 and h_a =
      // X_phiaphi / r^2; W_i^kn = X^k_mi g^mn
      const double Hr = dH.r, Hz = dH.z;
      const double hr = 0.5 * Hr, hz = 0.5 * Hz, Fr = r * lambda - hr, Fz = C - hz;
      const double Wr_rr = X.Urr * gA + X.Urz * rgC, Wr_rz = X.Urr * rgC + X.Urz * gB;
      const double Wr_zr = X.Vrr * gA + X.Vrz * rgC, Wr_zz = X.Vrr * rgC + X.Vrz * gB;
      const double Wz_rr = X.Urz * gA + X.Uzz * rgC, Wz_rz = X.Urz * rgC + X.Uzz * gB;
      const double Wz_zr = X.Vrz * gA + X.Vzz * rgC, Wz_zz = X.Vrz * rgC + X.Vzz * gB;
      RA += 3.0 * X.Prr * Wr_rr + X.Prz * (3.0 * Wr_rz + 2.0 * Wr_zr) + 2.0 * X.Pzz * Wr_zz + X.Qrr * Wr_zr +
            X.Qrz * Wr_zz + gH2 * hr * (2.0 * Fr + hr);
      RB += 3.0 * X.Qzz * Wz_zz + X.Qrz * (3.0 * Wz_zr + 2.0 * Wz_rz) + 2.0 * X.Qrr * Wz_rr + X.Prz * Wz_rr +
            X.Pzz * Wz_rz + gH2 * hz * (2.0 * Fz + hz);
      RC += (X.Qrr * Wr_rr + X.Qrz * (Wr_rz + 2.0 * Wr_zr) + 2.0 * X.Qzz * Wr_zz + X.Prr * Wz_rr +
             X.Prz * (Wz_rz + Wz_zr) + X.Pzz * Wz_zz + X.Prz * Wr_rr + X.Pzz * Wr_rz +
             gH2 * (hr * Fz + hz * (Fr + hr))) * ir;
      RH += -gC * Hz - r * g_lambda * Hr;
      RH += (-0.5 * C * gC * gH * Hr + gH * gC * Hz * Hr) * r + 0.5 * gH * Hz * Hz * gB + 1.5 * gC * Hz
            + 0.5 * gH * gA * Hr * Hr - 0.5 * C * gB * gH * Hz - 0.5 * gH * A * gC * Hz - C * gC - 0.5 * gC * Hz
            + 0.5 * (2.0 * gA - gH - gH * A * gA) * Hr * ir + gH * lambda * (1.0 - gA * H);
    }
    part(RA, RB, RC, RH, X.Urr, X.Urz, X.Uzz, X.Vrr, X.Vrz, X.Vzz);
    // the conformal factor's part
    double Drp, Dzp, RSCAL;
    {
      D2 dp;
      if constexpr (PHIMODE) {
        dp = hess<IN>(Fphi, G, W, i, j);
      } else {
        const D2 dc = hess<IN>(Fchi, G, W, i, j);
        const double qr = dc.r * ic, qz = dc.z * ic;
        dp.r = -0.5 * qr;
        dp.z = -0.5 * qz;
        dp.rr = -0.5 * (dc.rr * ic - qr * qr);
        dp.zz = -0.5 * (dc.zz * ic - qz * qz);
        dp.rz = -0.5 * (dc.rz * ic - qr * qz);
      }
      Drp = dp.r;
      Dzp = dp.z;
      double PA = -2.0 * (dp.rr - X.Urr * Drp - X.Vrr * Dzp);
      double PB = -2.0 * (dp.zz - X.Uzz * Drp - X.Vzz * Dzp);
      double PC = -2.0 * (dp.rz - X.Urz * Drp - X.Vrz * Dzp) * ir;
      const double PH = -2.0 * hess_H(Drp, Dzp, dH, r, ir, H, gA, gB, gC);
      const double aux = gA * PA + gB * PB + gH * PH + 2.0 * r2 * gC * PC
                         - 4.0 * (gA * Drp * Drp + gB * Dzp * Dzp + 2.0 * rgC * Drp * Dzp);
      PA += 4.0 * Drp * Drp;
      PB += 4.0 * Dzp * Dzp;
      PC += 4.0 * Drp * Dzp * ir;
      RA += PA + A * aux;
      RB += PB + B * aux;
      RH += PH + H * aux;
      RC += PC + C * aux;
      RSCAL = (gA * RA + gB * RB + gH * RH + 2.0 * r2 * gC * RC) * ipsi4;
    }
    {
      part(RA, RB, RC, RSCAL, Drp, Dzp);
      // D_i D_j alpha and its trace (:1268-1324)
      double sKA, sKB, sKC, Lapla;
      {
        const D2 da = hess<IN>(Fa, G, W, i, j);
        const double Dra = da.r, Dza = da.z;
        double d2A = da.rr - X.Urr * Dra - X.Vrr * Dza;
        double d2B = da.zz - X.Uzz * Dra - X.Vzz * Dza;
        double d2H = hess_H(Dra, Dza, dH, r, ir, H, gA, gB, gC);
        double d2C = (da.rz - X.Urz * Dra - X.Vrz * Dza) * ir;
        const double aux = gA * Dra * Drp + gB * Dza * Dzp + rgC * (Dra * Dzp + Dza * Drp);
        d2A -= 2.0 * (2.0 * Dra * Drp - A * aux);
        d2B -= 2.0 * (2.0 * Dza * Dzp - B * aux);
        d2H += 2.0 * H * aux;
        d2C -= 2.0 * (Dra * ir * Dzp + Dza * Drp * ir - C * aux);
        Lapla = (gA * d2A + gB * d2B + gH * d2H + 2.0 * r2 * gC * d2C) * ipsi4;
        const double tr = -Lapla + alpha * RSCAL;
        sKA = (-d2A + alpha * RA) * ipsi4 - third * A * tr;
        sKB = (-d2B + alpha * RB) * ipsi4 - third * B * tr;
        sKC = (-d2C + alpha * RC) * ipsi4 - third * C * tr;
      }
      part(sKA, sKB, sKC, Lapla);
      // quadratic terms of the extrinsic curvature (:970-1050)
      double strK;
      const double trK = FK(i, j);
      {
        const double KTA = FKA(i, j), KTB = FKB(i, j), KTC = FKC(i, j);
        const double KTH = -(gA * KTA + gB * KTB + 2.0 * r2 * gC * KTC) * H;
        const double KT2_A = (2.0 * KTA * gC * KTC + KTC * KTC * gB) * r2 + gA * KTA * KTA;
        const double KT2_B = (KTC * KTC * gA + 2.0 * KTC * gC * KTB) * r2 + gB * KTB * KTB;
        const double KT2_H = KTH * KTH * gH;
        const double KT2_C = KTC * KTC * gC * r2 + KTA * gA * KTC + KTA * gC * KTB + KTC * gB * KTB;
        const double KT2 = gA * KT2_A + gB * KT2_B + gH * KT2_H + 2.0 * gC * KT2_C * r2;
        strK = -Lapla + alpha * (KT2 + third * trK * trK);
        sKA += alpha * (trK * KTA - 2.0 * KT2_A);
        sKB += alpha * (trK * KTB - 2.0 * KT2_B);
        sKC += alpha * (trK * KTC - 2.0 * KT2_C);
      }
      if constexpr (SCALAR) {
        const Matter m = matter_point<SHIFT>(P, V, i, j, r, ir, A, B, H, C, gA, gB, gH, gC, ipsi4, ic * ic);
        strK += 4.0 * smallpi * alpha * (m.rho + m.trS);
        sKA -= 8.0 * smallpi * alpha * (m.S_A * ipsi4 - third * A * m.trS);
        sKB -= 8.0 * smallpi * alpha * (m.S_B * ipsi4 - third * B * m.trS);
        sKC -= 8.0 * smallpi * alpha * (m.S_C * ipsi4 - third * C * m.trS);
      }
      if constexpr (SHIFT) {
        part(strK, sKA, sKB, sKC);
        const D1 dbr = grad<IN>(fld(shift_slot(SH_beta_r)), G, W, i, j);
        const D1 dbz = grad<IN>(fld(shift_slot(SH_beta_z)), G, W, i, j);
        const double div = dbr.r + dbz.z + br * ir;
        const double KTA = FKA(i, j), KTB = FKB(i, j), KTC = FKC(i, j);
        sKA += 2.0 * (KTA * dbr.r + r * KTC * dbz.r) - t23 * KTA * div;
        sKB += 2.0 * (KTB * dbz.z + r * KTC * dbr.z) - t23 * KTB * div;
        sKC += KTC * br * ir + KTC * (dbr.r + dbz.z) + (KTB * dbz.r + KTA * dbr.z) * ir - t23 * KTC * div;
      }
      part(sKA, sKB, sKC);
      const int slot[4] = {S_trK, S_KTA, S_KTB, S_KTC};
      const RkUpdate<4> rk(S, yp, acc, slot, pl, k);
      strK += advko(FK);
      if (P.slicing == OA_SLICING_MAXIMAL) strK = 0.0;
      part(strK);
      sKA += advko(FKA);
      part(sKA);
      sKB += advko(FKB);
      part(sKB);
      sKC += advko(FKC);
      // radiative boundaries on level 0 (radiative_geometry.f90:58-237)
      if (radiative) {
        const D1 dK = grad<IN>(FK, G, W, i, j), dKA = grad<IN>(FKA, G, W, i, j), dKB = grad<IN>(FKB, G, W, i, j);
        const D1 dKC = grad<IN>(FKC, G, W, i, j);
        const double irr = 1.0 / sqrt(r * r + z * z);
        const double va = sqrt(P.gauge_f);
        if (P.slicing != OA_SLICING_MAXIMAL) strK = -va * (r * dK.r + z * dK.z + trK) * irr;
        sKA = -(r * dKA.r + z * dKA.z + FKA(i, j)) * irr;
        sKB = -(r * dKB.r + z * dKB.z + FKB(i, j)) * irr;
        const double c = third * (1.0 - 1.0 / va);
        if (onr) { sKA += c * strK * 2.0; sKB -= c * strK; }
        if (onzL) { sKA -= c * strK; sKB += c * strK * 2.0; }
        if (onzR) { sKA -= c * strK; sKB += c * strK * 2.0; }
        sKC = -(r * dKC.r + z * dKC.z + FKC(i, j)) * irr;
      }
      put(yo + S_trK * pl, G, i, j, rk(0, S_trK * pl + k, strK), 1.0, 1.0);
      put(yo + S_KTA * pl, G, i, j, rk(1, S_KTA * pl + k, sKA), 1.0, 1.0);
      put(yo + S_KTB * pl, G, i, j, rk(2, S_KTB * pl + k, sKB), 1.0, 1.0);
      put(yo + S_KTC * pl, G, i, j, rk(3, S_KTC * pl + k, sKC), 1.0, -1.0);
      part();
    }
  }

  // ---- Delta and the shift (Gammadriver2)
  if constexpr ((ROLE & ROLE_DELTA) != 0) {
    const double Delta_r = FDr(i, j), Delta_z = FDz(i, j);
    const double KTA = FKA(i, j), KTB = FKB(i, j), KTC = FKC(i, j);
    const double gA2 = gA * gA, gB2 = gB * gB, gC2 = gC * gC;
    // contravariant KT (:970-1050)
    const double KTup_rr = (2.0 * gA * gC * KTC + gC2 * KTB) * r2 + gA2 * KTA;
    const double KTup_zz = (gC2 * KTA + 2.0 * gC * gB * KTC) * r2 + gB2 * KTB;
    const double KTup_rz = gC2 * (r2 * r) * KTC + (gC * gA * KTA + gB * gA * KTC + gB * gC * KTB) * r;
    double DIV_r, DIV_z, DIVA_r, DIVA_z;
    {
      // calc_DIVKTA.f90:573-636: D'_m KT^im = g^ik (Z_k - Y_k - Delta^l KT_kl)
      // with Z_k = g^ml D'_m KT_kl, Y_k = T_mkq KT^qm and the evolved Delta,
      // and D_m KT^im the same with T_kmq KT^qm / 2 in place of Y_k
      const double KTH = -(gA * KTA + gB * KTB + 2.0 * r2 * gC * KTC) * H;
      const double Kp = gH2 * KTH, rKC = r * KTC;
      double Zr = r * gH * ((KTA - KTH) * ir * ir) - (Delta_r * KTA + Delta_z * rKC);
      double Zz = gH * KTC - (Delta_r * rKC + Delta_z * KTB);
      double Yr = r * lambda * Kp, Yz = C * Kp, Tr, Tz;
      {
        const D1 d = grad<IN>(FA, G, W, i, j);
        Yr += d.r * KTup_rr + d.z * KTup_rz;
        Tr = 0.5 * (d.r * KTup_rr);
        Tz = 0.5 * (d.z * KTup_rr);
      }
      {
        const D1 d = grad<IN>(FB, G, W, i, j);
        Yz += d.r * KTup_rz + d.z * KTup_zz;
        Tr += 0.5 * (d.r * KTup_zz);
        Tz += 0.5 * (d.z * KTup_zz);
      }
      part(Yr, Yz, Tr, Tz);
      {
        const D1 d = grad<IN>(FH, G, W, i, j);
        Tr += 0.5 * (d.r * Kp);
        Tz += 0.5 * (d.z * Kp);
      }
      {
        const D1 d = grad<IN>(FC, G, W, i, j);
        const double Trz_r = C + r * d.r, Trz_z = r * d.z;
        Yr += Trz_r * KTup_rz + Trz_z * KTup_zz;
        Yz += Trz_r * KTup_rr + Trz_z * KTup_rz;
        Tr += Trz_r * KTup_rz;
        Tz += Trz_z * KTup_rz;
      }
      part(Yr, Yz, Tr, Tz);
      {
        const D1 d = grad<IN>(FKA, G, W, i, j);
        Zr += gA * d.r + rgC * d.z;
      }
      {
        const D1 d = grad<IN>(FKB, G, W, i, j);
        Zz += rgC * d.r + gB * d.z;
      }
      {
        const D1 d = grad<IN>(FKC, G, W, i, j);
        const double Kc_r = KTC + r * d.r, Kc_z = r * d.z;
        Zr += rgC * Kc_r + gB * Kc_z;
        Zz += gA * Kc_r + rgC * Kc_z;
      }
      DIV_r = gA * (Zr - Tr) + rgC * (Zz - Tz);
      DIV_z = rgC * (Zr - Tr) + gB * (Zz - Tz);
      DIVA_r = gA * (Zr - Yr) + rgC * (Zz - Yz);
      DIVA_z = rgC * (Zr - Yr) + gB * (Zz - Yz);
    }
    {
      part(DIV_r, DIV_z, DIVA_r, DIVA_z);
      const double eta = P.eta;
      double sDr, sDz;
      {
        const D1 da = grad<IN>(Fa, G, W, i, j);
        const D1 dp = grad_phi<PHIMODE, IN>(V, G, W, i, j, ic);
        const D1 dK = grad<IN>(FK, G, W, i, j);
        sDr = -2.0 * (KTup_rr * da.r + KTup_rz * da.z) - 2.0 * alpha * DIVA_r;
        sDr += eta * alpha * (DIV_r + 6.0 * (KTup_rr * dp.r + KTup_rz * dp.z) - t23 * (gA * dK.r + rgC * dK.z));
        sDz = -2.0 * (KTup_rz * da.r + KTup_zz * da.z) - 2.0 * alpha * DIVA_z;
        sDz += eta * alpha * (DIV_z + 6.0 * (KTup_rz * dp.r + KTup_zz * dp.z) - t23 * (rgC * dK.r + gB * dK.z));
      }
      if constexpr (SCALAR) {
        const double psi4 = ic * ic;
        const Matter m = matter_point<SHIFT>(P, V, i, j, r, ir, A, B, H, C, gA, gB, gH, gC, ipsi4, psi4);
        sDr -= 8.0 * smallpi * eta * alpha * m.J_r * psi4;
        sDz -= 8.0 * smallpi * eta * alpha * m.J_z * psi4;
      }
      if constexpr (SHIFT) {
        part(sDr, sDz);
        // second derivatives of the shift (:587-737), one component at a time
        const auto Fbr = fld(shift_slot(SH_beta_r)), Fbz = fld(shift_slot(SH_beta_z));
        double div, Dr_div, Dz_div;
        {
          const D2 d = hess<IN>(Fbr, G, W, i, j);
          double DDrr;
          if constexpr (IN) {
            DDrr = W.r12 * (8.0 * (Fbr(i + 1, j) * V.inv_r(1) - Fbr(i - 1, j) * V.inv_r(-1))
                            - (Fbr(i + 2, j) * V.inv_r(2) - Fbr(i - 2, j) * V.inv_r(-2)));
          } else {
            auto fbr_r = [&](int ii, int jj) { return Fbr(ii, jj) / ((static_cast<double>(ii) - 0.5) * G.dr); };
            DDrr = s_d1r(fbr_r, G, i, j);
          }
          div = d.r + br * ir;
          Dr_div = d.rr + DDrr;
          Dz_div = d.rz + d.z * ir;
          sDr += -Delta_r * d.r - Delta_z * d.z;
          sDr += 2.0 * rgC * d.rz + gA * d.rr + gB * d.zz + gH * DDrr;
        }
        part(sDr, Dr_div, Dz_div, div);
        {
          const D2 d = hess<IN>(Fbz, G, W, i, j);
          div += d.z;
          Dr_div += d.rz;
          Dz_div += d.zz;
          sDz += -Delta_r * d.r - Delta_z * d.z;
          sDz += 2.0 * rgC * d.rz + gA * d.rr + gB * d.zz + gH * d.r * ir;
        }
        sDr += third * (gA * Dr_div + rgC * Dz_div + 2.0 * Delta_r * div);
        sDz += third * (rgC * Dr_div + gB * Dz_div + 2.0 * Delta_z * div);
      }
      part(sDr, sDz);
      if constexpr (SHIFT) {
        constexpr int sbr_ = shift_slot(SH_beta_r), sbz_ = shift_slot(SH_beta_z);
        constexpr int sdr_ = shift_slot(SH_dtbeta_r), sdz_ = shift_slot(SH_dtbeta_z);
        const int slot[6] = {S_Delta_r, S_Delta_z, sbr_, sbz_, sdr_, sdz_};
        const RkUpdate<6> rk(S, yp, acc, slot, pl, k);
        sDr += advko(FDr);
        part(sDr);
        sDz += advko(FDz);
        const double dbr = fld(sdr_)(i, j), dbz = fld(sdz_)(i, j);
        double sbr = dbr, sbz = dbz;
        double sdbr = P.drivercsi * sDr, sdbz = P.drivercsi * sDz;
        if (P.driveradv) {
          // the advective derivatives of sources_shift.f90:229-280 are the DA*
          // arrays: upwinded with shiftadvect, the centred ones otherwise;
          // dtbeta is differentiated from the planes of S.dtb_pre if given
          const bool pre = S.dtb_pre != nullptr;
          sbr += adv(fld(sbr_));
          sbz += adv(fld(sbz_));
          part(sbr, sbz);
          sdbr += adv(V.dtb(0, pre)) - adv(FDr);
          part(sdbr);
          sdbz += adv(V.dtb(1, pre)) - adv(FDz);
        }
        sdbr -= P.drivereta * dbr;
        sdbz -= P.drivereta * dbz;
        if (radiative && P.drivercsi != 0.0) {
          const bool pre = S.dtb_pre != nullptr;
          const double irr = 1.0 / sqrt(r * r + z * z);
          const double vs = sqrt(4.0 * third * P.drivercsi);
          const D1 ddr = grad<IN>(V.dtb(0, pre), G, W, i, j);
          const D1 ddz = grad<IN>(V.dtb(1, pre), G, W, i, j);
          sdbr = -vs * (r * ddr.r + z * ddr.z + dbr) * irr;
          sdbz = -vs * (r * ddz.r + z * ddz.z + dbz) * irr;
        }
        if (!pt0) {
          put(yo + S_Delta_r * pl, G, i, j, rk(0, S_Delta_r * pl + k, sDr), -1.0, 1.0);
          put(yo + S_Delta_z * pl, G, i, j, rk(1, S_Delta_z * pl + k, sDz), 1.0, -1.0);
        }
        put(yo + sbr_ * pl, G, i, j, rk(2, sbr_ * pl + k, sbr), -1.0, 1.0);
        put(yo + sbz_ * pl, G, i, j, rk(3, sbz_ * pl + k, sbz), 1.0, -1.0);
        put(yo + sdr_ * pl, G, i, j, rk(4, sdr_ * pl + k, sdbr), -1.0, 1.0);
        put(yo + sdz_ * pl, G, i, j, rk(5, sdz_ * pl + k, sdbz), 1.0, -1.0);
      } else if (!pt0) {
        const int slot[2] = {S_Delta_r, S_Delta_z};
        const RkUpdate<2> rk(S, yp, acc, slot, pl, k);
        sDr += advko(FDr);
        part(sDr);
        sDz += advko(FDz);
        put(yo + S_Delta_r * pl, G, i, j, rk(0, S_Delta_r * pl + k, sDr), -1.0, 1.0);
        put(yo + S_Delta_z * pl, G, i, j, rk(1, S_Delta_z * pl + k, sDz), 1.0, -1.0);
      }
      part();
    }
  }

  // ---- lapse (first-order Bona-Masso) and conformal factor, lagrangian:
  // sigma = 1
  if constexpr ((ROLE & ROLE_LAPSE) != 0) {
    // chi or phi is evolved; the projection gives the other
    const bool by_phi = pt0 || !P.chimethod;
    const int sp = by_phi ? S_phi : S_chi;
    const int slot[2] = {S_alpha, sp};
    const RkUpdate<2> rk(S, yp, acc, slot, pl, k);
    const double trK = FK(i, j);
    double salpha = 0.0;
    if (P.slicing != OA_SLICING_STATIC && P.slicing != OA_SLICING_MAXIMAL) {
      double falpha;
      if (P.slicing == OA_SLICING_HARMONIC) falpha = alpha * alpha * P.gauge_f;
      else if (P.slicing == OA_SLICING_1PLUSLOG) falpha = alpha * P.gauge_f;
      else falpha = alpha * alpha + (P.gauge_f - 1.0);
      salpha = -falpha * trK;
      if constexpr (SHIFT) salpha += adv(Fa);
      if (P.gauge_eta != 0.0) salpha -= P.gauge_eta * log(fabs(alpha));
    }
    double sphi = -alpha * trK / 6.0;
    double schi = 2.0 / 6.0 * alpha * chi * trK;
    if constexpr (SHIFT) {
      part(salpha, sphi, schi);
      double div = s_d1<IN, 0>(fld(shift_slot(SH_beta_r)), G, W, i, j) +
                   s_d1<IN, 1>(fld(shift_slot(SH_beta_z)), G, W, i, j) + br * ir;
      double a_phi, a_chi = 0.0;
      if constexpr (PHIMODE) {
        a_phi = adv(Fphi);
      } else {
        a_chi = adv(Fchi);
        a_phi = -0.5 * a_chi * ic;
      }
      sphi += a_phi + div / 6.0;
      schi += a_chi - 2.0 / 6.0 * chi * div;
    }
    Proj q;
    const double alpha_n = rk(0, S_alpha * pl + k, salpha);
    const double cf = rk(1, sp * pl + k, by_phi ? sphi : schi);
    q.phi = by_phi ? cf : 0.0;
    q.chi = by_phi ? chi : cf;
    project_factor(q, pt0, P.chimethod, SCALAR);
    put(yo + S_alpha * pl, G, i, j, alpha_n, 1.0, 1.0);
    put(yo + S_chi * pl, G, i, j, q.chi, 1.0, 1.0);
    if (by_phi) put(yo + S_phi * pl, G, i, j, q.phi, 1.0, 1.0);
    part();
  }

  // ---- conformal metric
  if constexpr ((ROLE & ROLE_METRIC) != 0) {
    const int slot[4] = {S_A, S_B, S_H, S_C};
    const RkUpdate<4> rk(S, yp, acc, slot, pl, k);
    const double KTA = FKA(i, j), KTB = FKB(i, j), KTC = FKC(i, j);
    const double KTH = -(gA * KTA + gB * KTB + 2.0 * r2 * gC * KTC) * H;
    double sA = -2.0 * alpha * KTA, sB = -2.0 * alpha * KTB, sH = -2.0 * alpha * KTH, sC = -2.0 * alpha * KTC;
    if constexpr (SHIFT) {
      const D1 dbr = grad<IN>(fld(shift_slot(SH_beta_r)), G, W, i, j);
      const D1 dbz = grad<IN>(fld(shift_slot(SH_beta_z)), G, W, i, j);
      const double div = dbr.r + dbz.z + br * ir;
      sA += 2.0 * (A * dbr.r + r * C * dbz.r) - t23 * A * div;
      sB += 2.0 * (B * dbz.z + r * C * dbr.z) - t23 * B * div;
      sH += 2.0 * H * br * ir - t23 * H * div;
      sC += C * br * ir + C * (dbr.r + dbz.z) + (B * dbz.r + A * dbr.z) * ir - t23 * C * div;
      part(sA, sB, sH, sC);
      sA += adv(FA);
      part(sA);
      sB += adv(FB);
      part(sB);
      sH += adv(FH);
      part(sH);
      sC += adv(FC);
    }
    Proj q;
    q.A = rk(0, S_A * pl + k, sA);
    q.B = rk(1, S_B * pl + k, sB);
    q.H = rk(2, S_H * pl + k, sH);
    q.C = rk(3, S_C * pl + k, sC);
    if (!pt0) factordet(q, r);
    put(yo + S_A * pl, G, i, j, q.A, 1.0, 1.0);
    put(yo + S_B * pl, G, i, j, q.B, 1.0, 1.0);
    put(yo + S_H * pl, G, i, j, q.H, 1.0, 1.0);
    put(yo + S_C * pl, G, i, j, q.C, 1.0, -1.0);
    part();
  }

  // ---- the real scalar field (scalar.f90:94-251)
  if constexpr (SCALAR && (ROLE & ROLE_SCALAR) != 0) {
    constexpr int s0 = scalar_slot(SHIFT, SC_phi), s1 = scalar_slot(SHIFT, SC_xi_r);
    constexpr int s2 = scalar_slot(SHIFT, SC_xi_z), s3 = scalar_slot(SHIFT, SC_pi);
    const auto Fsp = fld(s0), Fxr = fld(s1), Fxz = fld(s2), Fpi = fld(s3);
    const double xr = Fxr(i, j), xz = Fxz(i, j), pi = Fpi(i, j);
    const int slot[4] = {s0, s1, s2, s3};
    const RkUpdate<4> rk(S, yp, acc, slot, pl, k);
    // -(g^rr,r + r g^rz,z) and -(g^zz,z + r g^rz,r + g^rz)
    double Dd_r, Dd_z;
    deldef<IN>(V, G, W, i, j, r, gC, 0.0, Dd_r, Dd_z);
    const double mr = -Dd_r, mz = -Dd_z - gC;
    part(Dd_r, Dd_z);
    double dr_, dz_, spi;
    if (P.scalarmethod == OA_SCALARMETHOD_FIRST) {
      const D1 dxr = grad<IN>(Fxr, G, W, i, j), dxz = grad<IN>(Fxz, G, W, i, j);
      dr_ = xr; dz_ = xz;
      spi = alpha * (gA * dxr.r + gB * dxz.z + rgC * (dxz.r + dxr.z));
    } else {
      const D2 ds = hess<IN>(Fsp, G, W, i, j);
      dr_ = ds.r; dz_ = ds.z;
      spi = alpha * (gA * ds.rr + gB * ds.zz + 2.0 * rgC * ds.rz);
    }
    part(dr_, dz_, spi);
    const double ur = gA * dr_ + rgC * dz_, uz = gB * dz_ + rgC * dr_;
    const D1 dp = grad_phi<PHIMODE, IN>(V, G, W, i, j, ic);
    const D1 da = grad<IN>(Fa, G, W, i, j);
    spi += 2.0 * alpha * (dp.r * ur + dp.z * uz);
    spi += da.r * ur + da.z * uz;
    spi += alpha * (dr_ * mr + dz_ * mz);
    spi += alpha * (gA * dr_ * ir + gC * dz_);
    spi = spi * ipsi4;
    spi += alpha * pi * FK(i, j);
    if (P.scalarpotential != OA_POT_NONE) {
      const double ph = Fsp(i, j);
      double VP = P.scalar_mass * P.scalar_mass * ph;
      if (P.scalarpotential == OA_POT_PHI4) VP += P.scalar_lambda * ph * ph * ph;
      spi -= alpha * VP;
    }
    double s_sphi = alpha * pi, s_sxr = pi * da.r, s_sxz = pi * da.z;
    part(spi, s_sphi, s_sxr, s_sxz);
    if constexpr (SHIFT) {
      const D1 dbr = grad<IN>(fld(shift_slot(SH_beta_r)), G, W, i, j);
      const D1 dbz = grad<IN>(fld(shift_slot(SH_beta_z)), G, W, i, j);
      s_sphi += br * xr + bz * xz;
      s_sxr += xr * dbr.r + xz * dbz.r;
      s_sxz += xr * dbr.z + xz * dbz.z;
    }
    const D1 dpi = grad<IN>(Fpi, G, W, i, j);
    s_sxr += alpha * dpi.r;
    s_sxz += alpha * dpi.z;
    spi += advkos(Fpi);
    part(spi, s_sxr, s_sxz);
    s_sxr += advkos(Fxr);
    part(s_sxr);
    s_sxz += advkos(Fxz);
    part(s_sxz);
    s_sphi += advdis<IN, 0>(Fsp, G, P, W, i, j, br, bz, W.ko_s, sdis);
    // radiative boundary on pi at every level (scalar.f90:244-251)
    if (bnd) {
      const double rr = sqrt(r * r + z * z);
      spi = -(r * dpi.r + z * dpi.z + pi) / rr;
    }
    put(yo + s0 * pl, G, i, j, rk(0, s0 * pl + k, s_sphi), 1.0, 1.0);
    put(yo + s1 * pl, G, i, j, rk(1, s1 * pl + k, s_sxr), -1.0, 1.0);
    put(yo + s2 * pl, G, i, j, rk(2, s2 * pl + k, s_sxz), 1.0, -1.0);
    put(yo + s3 * pl, G, i, j, rk(3, s3 * pl + k, spi), 1.0, 1.0);
  }
}

}  // namespace oax
