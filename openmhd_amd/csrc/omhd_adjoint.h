// omhd_adjoint.h -- the per-cell and per-interface pieces of the step and
// their hand-written reverse (vector-Jacobian) forms, in plain C++ that
// compiles for the device (included by omhd_adjoint.hip) and for the host.
//
//   prim_fwd / prim_vjp   u2v at one cell          (2D_basic/u2v.f90:23-26)
//   lim_fwd  / lim_coef   slope limiter at one cell (2D_basic/limiter.f90)
//   hlld_fwd / hlld_vjp   HLLD flux at one face     (2D_basic/flux_solver.f90:352-585)
//
// The *_fwd forms are templates over the scalar type so that the same
// statements run in double (where they give the reference's bits: they follow
// its evaluation order) and in a dual-number type (forward-mode tangents, used
// to check every reverse form exactly).  Branch decisions are taken on values
// and recorded implicitly: the reverse forms recompute them from the same
// inputs, so the adjoint differentiates the branch the forward pass took, with
// one-sided derivatives at the kinks (|x| has slope +1 at x = 0, min(a, b)
// follows b on a tie, max(a, b) follows b on a tie, sqrt(max(q, 0)) has zero
// slope where its argument is 0, and SIGN(c, x) is constant).
#pragma once
#include <math.h>

#if defined(__HIPCC__)
#include "omhd_device.h"
#endif

#if defined(__HIPCC__)
#define OMHD_HD __host__ __device__ inline
#else
#define OMHD_HD inline
#endif

namespace omhd {
namespace adj {

constexpr double kGam = 5.0 / 3.0;  // param.h:3
constexpr int NV = 9;               // vx vy vz p | mx my mz en ; ro bx by bz psi

OMHD_HD double val(double a) { return a; }
OMHD_HD double tsqrt(double a) { return sqrt(a); }
OMHD_HD double tabs(double a) { return a < 0 ? -a : a; }
OMHD_HD double tmin(double a, double b) { return a < b ? a : b; }
OMHD_HD double tmax(double a, double b) { return a > b ? a : b; }
// Fortran SIGN(c, x) for a constant magnitude c: copysign semantics
template <class T>
OMHD_HD double csign(double c, const T &x) {
  return copysign(c, val(x));
}
OMHD_HD double slope_abs(double x) { return x < 0 ? -1.0 : 1.0; }  // d|x|/dx as tabs takes it

// ---------------------------------------------------------------------------
// u2v at one cell: u = (mx,my,mz,en,ro,bx,by,bz,psi) -> w = (vx,vy,vz,p,ro,B,psi)
// ---------------------------------------------------------------------------
template <class T>
OMHD_HD void prim_fwd(const T u[NV], T w[NV]) {
  const T rho = u[4];
  const T v1 = u[0] / rho, v2 = u[1] / rho, v3 = u[2] / rho;
  const T rv2 = v1 * u[0] + v2 * u[1] + v3 * u[2];
  const T B2 = u[5] * u[5] + u[6] * u[6] + u[7] * u[7];
  w[0] = v1;
  w[1] = v2;
  w[2] = v3;
  w[3] = (kGam - 1) * (u[3] - 0.5 * (rv2 + B2));
  for (int m = 4; m < NV; m++) w[m] = u[m];
}

// bu += (dw/du)^T bw, from the primitive values w of the cell (v = m/rho,
// p = (gam-1)(en - 0.5 (m.v + B.B)))
OMHD_HD void prim_vjp(const double w[NV], const double bw[NV], double bu[NV]) {
  const double rho = w[4], ir = 1.0 / rho;
  const double bp = (kGam - 1) * bw[3];
  const double brv2 = -0.5 * bp;
  const double v2 = w[0] * w[0] + w[1] * w[1] + w[2] * w[2];
  double brho = bw[4] - v2 * brv2;
  for (int m = 0; m < 3; m++) {
    bu[m] += bw[m] * ir + 2.0 * w[m] * brv2;
    brho -= bw[m] * w[m] * ir;
  }
  bu[3] += bp;
  bu[4] += brho;
  for (int m = 5; m < 8; m++) bu[m] += bw[m] - w[m] * bp;  // dB2 = 2B dB, times -0.5
  bu[8] += bw[8];
}

// ---------------------------------------------------------------------------
// Slope limiter at one cell from (w[c-1], w[c], w[c+1]): gR = w0 - gradR is the
// right state of the lower face, gL = w0 + gradL the left state of the upper
// face (limiter.f90: minmod :84-101, MC :141-158, van Leer :201-210, Koren
// :256-272; type 0 copies the cell value).
// ---------------------------------------------------------------------------
template <class T>
OMHD_HD void lim_fwd(int type, const T &wm, const T &w0, const T &wp, T &gR, T &gL) {
  if (type == 0) {
    gR = w0;
    gL = w0;
  } else if (type == 1) {
    const T gA = (w0 - wm), gB = (wp - w0);
    const T grad = (csign(0.25, gA) + csign(0.25, gB)) * tmin(tabs(gA), tabs(gB));
    gR = w0 - grad;
    gL = w0 + grad;
  } else if (type == 2) {
    const T gA = (w0 - wm), gB = (wp - w0);
    const T gC = 0.25 * (wp - wm);
    const T grad = (csign(0.5, gA) + csign(0.5, gB)) * tmin(tmin(tabs(gA), tabs(gB)), tabs(gC));
    gR = w0 - grad;
    gL = w0 + grad;
  } else if (type == 3) {
    const T gA = (w0 - wm), gB = (wp - w0);
    const T grad = (val(gA) * val(gB) <= 0) ? T(0.0) : gA * gB / (gA + gB);
    gR = w0 - grad;
    gL = w0 + grad;
  } else {
    const double f1 = 1.0 / 6.0;
    const T gA = (w0 - wm), gB = (wp - w0);
    const double s = csign(0.5, gA) + csign(0.5, gB);
    const T m = tmin(tabs(gA), tabs(gB));
    T gC = f1 * (2 * gA + gB);
    gR = w0 - s * tmin(m, tabs(gC));
    gC = f1 * (gA + 2 * gB);
    gL = w0 + s * tmin(m, tabs(gC));
  }
}

// Derivatives of gradR and gradL with respect to (wm, w0, wp):
// d gradR = cR[0] dwm + cR[1] dw0 + cR[2] dwp, likewise gradL.
OMHD_HD void lim_coef(int type, double wm, double w0, double wp, double cR[3], double cL[3]) {
  double kAR = 0, kBR = 0, kAL = 0, kBL = 0;  // d grad / d gA, d gB
  const double gA = (w0 - wm), gB = (wp - w0);
  if (type == 1 || type == 2) {
    const double s = (type == 1) ? csign(0.25, gA) + csign(0.25, gB) : csign(0.5, gA) + csign(0.5, gB);
    const double aA = tabs(gA), aB = tabs(gB);
    double kA = (aA < aB) ? s * slope_abs(gA) : 0.0;
    double kB = (aA < aB) ? 0.0 : s * slope_abs(gB);
    if (type == 2) {
      const double gC = 0.25 * (wp - wm);
      const double m1 = tmin(aA, aB);
      if (!(m1 < tabs(gC))) {  // the min picked |gC| = 0.25 |gB + gA|
        const double kC = s * slope_abs(gC) * 0.25;
        kA = kC;
        kB = kC;
      }
    }
    kAR = kAL = kA;
    kBR = kBL = kB;
  } else if (type == 3) {
    // by a select, as below
    const double S = gA + gB, iS2 = 1.0 / (S * S);
    kAR = kAL = gA * gB <= 0 ? 0.0 : gB * gB * iS2;
    kBR = kBL = gA * gB <= 0 ? 0.0 : gA * gA * iS2;
  } else if (type == 4) {
    const double f1 = 1.0 / 6.0;
    const double s = csign(0.5, gA) + csign(0.5, gB);
    const double aA = tabs(gA), aB = tabs(gB);
    const double mA = (aA < aB) ? slope_abs(gA) : 0.0, mB = (aA < aB) ? 0.0 : slope_abs(gB);
    const double m = tmin(aA, aB);
    const double c1 = f1 * (2 * gA + gB), c2 = f1 * (gA + 2 * gB);
    // by selects: branches here took a kernel with 81 of them out of its registers
    const bool i1 = m < tabs(c1), i2 = m < tabs(c2);
    const double u1 = s * slope_abs(c1) * f1, u2 = s * slope_abs(c2) * f1;
    kAR = i1 ? s * mA : 2 * u1;
    kBR = i1 ? s * mB : u1;
    kAL = i2 ? s * mA : u2;
    kBL = i2 ? s * mB : 2 * u2;
  }
  // gA = w0 - wm, gB = wp - w0
  cR[0] = -kAR;
  cR[1] = kAR - kBR;
  cR[2] = kBR;
  cL[0] = -kAL;
  cL[1] = kAL - kBL;
  cL[2] = kBL;
}

// ---------------------------------------------------------------------------
// HLLD flux at one interface, flux_solver.f90:352-585 (Miyoshi & Kusano 2005
// with the HLLC-G fallback of Gurski 2004).  D = dir - 1; L, R in the slot
// order (vx,vy,vz,p,ro,bx,by,bz,psi).  branch: 1 FL, 2 FR, 3/4 HLLC-G left /
// right of the contact, 5 L*, 6 R*, 7 L**, 8 R**.
// ---------------------------------------------------------------------------
template <int D, class T>
OMHD_HD void hlld_fwd(const T L[NV], const T R[NV], double ch, T F[NV], int *branch = nullptr) {
  constexpr int vn = D, vt1 = (D + 1) % 3, vt2 = (D + 2) % 3;
  constexpr int mn = vn, mt1 = vt1, mt2 = vt2;
  constexpr int bn = 5 + vn, bt1 = 5 + vt1, bt2 = 5 + vt2;
  constexpr int RO = 4, PR = 3, EN = 3, PS = 8;
  const double r1 = 1.0 / (kGam - 1.0), r2 = kGam / (kGam - 1.0), hllg = 1.001;
  T UL[4], UR[4], FL[NV], FR[NV];
  for (int m = 0; m < NV; m++) {
    FL[m] = T(0.0);
    FR[m] = T(0.0);
    F[m] = T(0.0);
  }
  int br = 0;
  T v2 = L[0] * L[0] + L[1] * L[1] + L[2] * L[2];
  T B2 = L[5] * L[5] + L[6] * L[6] + L[7] * L[7];
  const T vBL = L[0] * L[5] + L[1] * L[6] + L[2] * L[7];
  UL[0] = L[RO] * L[0];
  UL[1] = L[RO] * L[1];
  UL[2] = L[RO] * L[2];
  UL[EN] = 0.5 * (L[RO] * v2 + B2) + r1 * L[PR];
  FL[RO] = L[RO] * L[vn];
  FL[mn] = L[RO] * L[vn] * L[vn] - L[bn] * L[bn] + L[PR] + 0.5 * B2;
  FL[mt1] = L[RO] * L[vn] * L[vt1] - L[bn] * L[bt1];
  FL[mt2] = L[RO] * L[vn] * L[vt2] - L[bn] * L[bt2];
  FL[EN] = (0.5 * L[RO] * v2 + r2 * L[PR] + B2) * L[vn] - vBL * L[bn];
  FL[bt1] = L[vn] * L[bt1] - L[bn] * L[vt1];
  FL[bt2] = L[vn] * L[bt2] - L[bn] * L[vt2];
  T f1 = kGam * L[PR];
  T f2 = 4 * (L[bn] * L[bn]);
  T aL = ((f1 + B2) + tsqrt(tmax((f1 + B2) * (f1 + B2) - f1 * f2, T(0.0)))) / (2 * L[RO]);
  const T ptL = L[PR] + 0.5 * B2;

  v2 = R[0] * R[0] + R[1] * R[1] + R[2] * R[2];
  B2 = R[5] * R[5] + R[6] * R[6] + R[7] * R[7];
  const T vBR = R[0] * R[5] + R[1] * R[6] + R[2] * R[7];
  UR[0] = R[RO] * R[0];
  UR[1] = R[RO] * R[1];
  UR[2] = R[RO] * R[2];
  UR[EN] = 0.5 * (R[RO] * v2 + B2) + r1 * R[PR];
  FR[RO] = R[RO] * R[vn];
  FR[mn] = R[RO] * R[vn] * R[vn] - R[bn] * R[bn] + R[PR] + 0.5 * B2;
  FR[mt1] = R[RO] * R[vn] * R[vt1] - R[bn] * R[bt1];
  FR[mt2] = R[RO] * R[vn] * R[vt2] - R[bn] * R[bt2];
  FR[EN] = (0.5 * R[RO] * v2 + r2 * R[PR] + B2) * R[vn] - vBR * R[bn];
  FR[bt1] = R[vn] * R[bt1] - R[bn] * R[vt1];
  FR[bt2] = R[vn] * R[bt2] - R[bn] * R[vt2];
  f1 = kGam * R[PR];
  f2 = 4 * (R[bn] * R[bn]);
  T aR = ((f1 + B2) + tsqrt(tmax((f1 + B2) * (f1 + B2) - f1 * f2, T(0.0)))) / (2 * R[RO]);
  const T ptR = R[PR] + 0.5 * B2;

  f1 = tsqrt(tmax(aL, aR));
  aL = tmin(L[vn], R[vn]) - f1;
  aR = tmax(L[vn], R[vn]) + f1;

  if (val(aL) >= 0) {
    for (int m = 0; m < NV; m++) F[m] = FL[m];
    br = 1;
  } else if (val(aR) <= 0) {
    for (int m = 0; m < NV; m++) F[m] = FR[m];
    br = 2;
  } else {
    T Uh[NV];
    f1 = 1.0 / (aR - aL);
    for (int m = 0; m < 3; m++) Uh[m] = f1 * (aR * UR[m] - aL * UL[m] - FR[m] + FL[m]);
    for (int m = RO; m <= 7; m++) Uh[m] = f1 * (aR * R[m] - aL * L[m] - FR[m] + FL[m]);
    const T aM = Uh[mn] / Uh[RO];
    const T pt = ptL + L[RO] * (aL - L[vn]) * (aM - L[vn]);
    const T roL = L[RO] * (aL - L[vn]) / (aL - aM);
    const T roR = R[RO] * (aR - R[vn]) / (aR - aM);
    const T aVL = tabs(Uh[bn]) / tsqrt(roL);
    const T aVR = tabs(Uh[bn]) / tsqrt(roR);
    if ((val(aL) >= val(aM - hllg * aVL)) || (val(aM + hllg * aVR) >= val(aR))) {
      f2 = aL * aR;
      F[bt1] = f1 * (aR * FL[bt1] - aL * FR[bt1] + f2 * (R[bt1] - L[bt1]));
      F[bt2] = f1 * (aR * FL[bt2] - aL * FR[bt2] + f2 * (R[bt2] - L[bt2]));
      const T at1 = Uh[mt1] / Uh[RO];
      const T at2 = Uh[mt2] / Uh[RO];
      const T enL = ((aL - L[vn]) * UL[EN] - ptL * L[vn] + pt * aM +
                     Uh[bn] * (vBL - aM * Uh[bn] - at1 * Uh[bt1] - at2 * Uh[bt2])) / (aL - aM);
      const T enR = ((aR - R[vn]) * UR[EN] - ptR * R[vn] + pt * aM +
                     Uh[bn] * (vBR - aM * Uh[bn] - at1 * Uh[bt1] - at2 * Uh[bt2])) / (aR - aM);
      const double s1 = 0.5 + csign(0.5, aM);
      const double s2 = 1.0 - s1;
      F[mn] = s1 * (aL * (roL * aM - UL[mn]) + FL[mn]) + s2 * (aR * (roR * aM - UR[mn]) + FR[mn]);
      F[mt1] = s1 * (aL * (roL * at1 - UL[mt1]) + FL[mt1]) + s2 * (aR * (roR * at1 - UR[mt1]) + FR[mt1]);
      F[mt2] = s1 * (aL * (roL * at2 - UL[mt2]) + FL[mt2]) + s2 * (aR * (roR * at2 - UR[mt2]) + FR[mt2]);
      F[EN] = s1 * (aL * (enL - UL[EN]) + FL[EN]) + s2 * (aR * (enR - UR[EN]) + FR[EN]);
      F[RO] = s1 * (aL * (roL - L[RO]) + FL[RO]) + s2 * (aR * (roR - R[RO]) + FR[RO]);
      br = (val(aM) >= 0) ? 3 : 4;
    } else {
      T UL1[NV], UR1[NV];
      f1 = 1.0 / (L[RO] * (aL - L[vn]) * (aL - aM) - Uh[bn] * Uh[bn]);
      UL1[bt1] = L[bt1] * f1 * (L[RO] * ((aL - L[vn]) * (aL - L[vn])) - Uh[bn] * Uh[bn]);
      UL1[bt2] = L[bt2] * f1 * (L[RO] * ((aL - L[vn]) * (aL - L[vn])) - Uh[bn] * Uh[bn]);
      const T vt1L = L[vt1] - f1 * Uh[bn] * L[bt1] * (aM - L[vn]);
      const T vt2L = L[vt2] - f1 * Uh[bn] * L[bt2] * (aM - L[vn]);
      UL1[RO] = roL;
      UL1[EN] = ((aL - L[vn]) * UL[EN] - ptL * L[vn] + pt * aM +
                 Uh[bn] * (vBL - aM * Uh[bn] - vt1L * UL1[bt1] - vt2L * UL1[bt2])) / (aL - aM);
      UL1[mn] = roL * aM;
      UL1[mt1] = roL * vt1L;
      UL1[mt2] = roL * vt2L;
      f1 = 1.0 / (R[RO] * (aR - R[vn]) * (aR - aM) - Uh[bn] * Uh[bn]);
      UR1[bt1] = R[bt1] * f1 * (R[RO] * ((aR - R[vn]) * (aR - R[vn])) - Uh[bn] * Uh[bn]);
      UR1[bt2] = R[bt2] * f1 * (R[RO] * ((aR - R[vn]) * (aR - R[vn])) - Uh[bn] * Uh[bn]);
      const T vt1R = R[vt1] - f1 * Uh[bn] * R[bt1] * (aM - R[vn]);
      const T vt2R = R[vt2] - f1 * Uh[bn] * R[bt2] * (aM - R[vn]);
      UR1[RO] = roR;
      UR1[EN] = ((aR - R[vn]) * UR[EN] - ptR * R[vn] + pt * aM +
                 Uh[bn] * (vBR - aM * Uh[bn] - vt1R * UR1[bt1] - vt2R * UR1[bt2])) / (aR - aM);
      UR1[mn] = roR * aM;
      UR1[mt1] = roR * vt1R;
      UR1[mt2] = roR * vt2R;
      const T aL1 = aM - aVL;
      const T aR1 = aM + aVR;
      if (val(aL1) >= 0) {
        for (int m = 0; m < 4; m++) F[m] = aL * (UL1[m] - UL[m]) + FL[m];
        F[RO] = aL * (UL1[RO] - L[RO]) + FL[RO];
        F[bt1] = aL * (UL1[bt1] - L[bt1]) + FL[bt1];
        F[bt2] = aL * (UL1[bt2] - L[bt2]) + FL[bt2];
        br = 5;
      } else if (val(aR1) <= 0) {
        for (int m = 0; m < 4; m++) F[m] = aR * (UR1[m] - UR[m]) + FR[m];
        F[RO] = aR * (UR1[RO] - R[RO]) + FR[RO];
        F[bt1] = aR * (UR1[bt1] - R[bt1]) + FR[bt1];
        F[bt2] = aR * (UR1[bt2] - R[bt2]) + FR[bt2];
        br = 6;
      } else {
        T U2[NV];
        const T roLs = tsqrt(roL);
        const T roRs = tsqrt(roR);
        f1 = 1.0 / (roLs + roRs);
        const double sB = csign(1.0, Uh[bn]);
        const T at1 = f1 * (roLs * vt1L + roRs * vt1R + (UR1[bt1] - UL1[bt1]) * sB);
        const T at2 = f1 * (roLs * vt2L + roRs * vt2R + (UR1[bt2] - UL1[bt2]) * sB);
        U2[bt1] = f1 * (roLs * UR1[bt1] + roRs * UL1[bt1] + roLs * roRs * (vt1R - vt1L) * sB);
        U2[bt2] = f1 * (roLs * UR1[bt2] + roRs * UL1[bt2] + roLs * roRs * (vt2R - vt2L) * sB);
        if (val(aM) >= 0) {
          U2[RO] = roL;
          U2[EN] = UL1[EN] - roLs * (vt1L * UL1[bt1] + vt2L * UL1[bt2] - at1 * U2[bt1] - at2 * U2[bt2]) * sB;
          U2[mn] = roL * aM;
          U2[mt1] = roL * at1;
          U2[mt2] = roL * at2;
          for (int m = 0; m < 4; m++) F[m] = aL1 * U2[m] - (aL1 - aL) * UL1[m] - aL * UL[m] + FL[m];
          F[RO] = aL1 * U2[RO] - (aL1 - aL) * UL1[RO] - aL * L[RO] + FL[RO];
          F[bt1] = aL1 * U2[bt1] - (aL1 - aL) * UL1[bt1] - aL * L[bt1] + FL[bt1];
          F[bt2] = aL1 * U2[bt2] - (aL1 - aL) * UL1[bt2] - aL * L[bt2] + FL[bt2];
          br = 7;
        } else {
          U2[RO] = roR;
          U2[EN] = UR1[EN] + roRs * (vt1R * UR1[bt1] + vt2R * UR1[bt2] - at1 * U2[bt1] - at2 * U2[bt2]) * sB;
          U2[mn] = roR * aM;
          U2[mt1] = roR * at1;
          U2[mt2] = roR * at2;
          for (int m = 0; m < 4; m++) F[m] = aR1 * U2[m] - (aR1 - aR) * UR1[m] - aR * UR[m] + FR[m];
          F[RO] = aR1 * U2[RO] - (aR1 - aR) * UR1[RO] - aR * R[RO] + FR[RO];
          F[bt1] = aR1 * U2[bt1] - (aR1 - aR) * UR1[bt1] - aR * R[bt1] + FR[bt1];
          F[bt2] = aR1 * U2[bt2] - (aR1 - aR) * UR1[bt2] - aR * R[bt2] + FR[bt2];
          br = 8;
        }
      }
    }
  }
  F[bn] = 0.5 * ((L[PS] + R[PS]) - ch * (R[bn] - L[bn]));
  F[PS] = 0.5 * (ch * ch * (L[bn] + R[bn]) - ch * (R[PS] - L[PS]));
  if (branch) *branch = br;
}

// ---------------------------------------------------------------------------
// Reverse of hlld_fwd.  Only the quantities its branches are decided by repeat
// hlld_fwd's statements bit for bit; what only the reverse needs is left to
// fused multiply-adds and plain reciprocals.
//
// Every side S enters the flux through FS - e US (its physical flux and e, the
// fan speed where a star state follows it and 0 where it does not) and through
// its star state.  The intermediate state Uh = iw (aR UR - aL UL - FR + FL)
// has the same form, so with
//   t_S[m] = [side S is taken] bF[m] +- iw bUh[m]        (+ for L, - for R)
// one side function reverses (FS - e US) . t_S, the flux's and Uh's parts at
// once, and the fan speeds get -US . t_S; no adjoints of FL, FR, UL and UR are
// kept.  Uh and iw need no flux either: biw / iw = Uh . bUh.
// ---------------------------------------------------------------------------
#if defined(__clang__)
#define OMHD_CONTRACT _Pragma("clang fp contract(fast)")
#else
#define OMHD_CONTRACT
#endif

// 1/x to an ulp, of any x: the fix-up gives what zeros, infinities and NaN give
// and what over- and underflow, so unlike quot's its uses need no range.  (The
// bits of 1.0 / x on 512 random values at each exponent, subnormals included.)
OMHD_HD double rinv(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_div_fixup(recip(x), x, 1.0);
#else
  return 1.0 / x;
#endif
}
// sqrt(x), correctly rounded
OMHD_HD double root(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return csqrt(x);
#else
  return sqrt(x);
#endif
}

// the side's quantities that hlld_fwd forms before the fans, and Uh's share
// aS US - FS of its three momenta, density and transverse field
template <int D>
struct SideFwd {
  double E, pt, vB, af;  // US[EN], total pressure, v.B, squared fast speed
  double F[NV];          // FS[mn], [mt1], [mt2], [RO], [bt1], [bt2]
};
template <int D>
OMHD_HD void side_fwd(const double S[NV], SideFwd<D> &o) {
  constexpr int vn = D, vt1 = (D + 1) % 3, vt2 = (D + 2) % 3;
  constexpr int bn = 5 + vn, bt1 = 5 + vt1, bt2 = 5 + vt2;
  constexpr int RO = 4, PR = 3;
  const double r1 = 1.0 / (kGam - 1.0);
  const double v2 = S[0] * S[0] + S[1] * S[1] + S[2] * S[2];
  const double B2 = S[5] * S[5] + S[6] * S[6] + S[7] * S[7];
  o.vB = S[0] * S[5] + S[1] * S[6] + S[2] * S[7];
  o.E = 0.5 * (S[RO] * v2 + B2) + r1 * S[PR];
  o.F[RO] = S[RO] * S[vn];
  o.F[vn] = S[RO] * S[vn] * S[vn] - S[bn] * S[bn] + S[PR] + 0.5 * B2;
  o.F[vt1] = S[RO] * S[vn] * S[vt1] - S[bn] * S[bt1];
  o.F[vt2] = S[RO] * S[vn] * S[vt2] - S[bn] * S[bt2];
  o.F[bt1] = S[vn] * S[bt1] - S[bn] * S[vt1];
  o.F[bt2] = S[vn] * S[bt2] - S[bn] * S[vt2];
  o.F[bn] = 0.0;
  const double f1 = kGam * S[PR], f2 = 4 * (S[bn] * S[bn]);
  o.af = ((f1 + B2) + root(tmax((f1 + B2) * (f1 + B2) - f1 * f2, 0.0))) / (2 * S[RO]);
  o.pt = S[PR] + 0.5 * B2;
}

// bs += the reverse of (FS - e US) . t, of pt, vB and US[EN] with the adjoints
// bpt, bvB and bE (e held), and of the squared fast speed af with ba
template <int D>
OMHD_HD void side_vjp(const double s[NV], const double t[NV], double e, double E, double pt, double vB, double af,
                      double ba, double bpt, double bvB, double bE, double bs[NV]) {
  OMHD_CONTRACT
  constexpr int vn = D, vt1 = (D + 1) % 3, vt2 = (D + 2) % 3;
  constexpr int bn = 5 + vn, bt1 = 5 + vt1, bt2 = 5 + vt2;
  constexpr int RO = 4, PR = 3, EN = 3;
  const double r1 = 1.0 / (kGam - 1.0);
  // FS - e US, with c = vn - e: ro c (1, v) [density, momenta], mn: - bn^2 + pt,
  // mt: - bn bt, bt: bt c - bn vt, en: E c + pt vn - bn vB
  const double c = s[vn] - e, rc = s[RO] * c, tE = t[EN];
  const double dot = s[0] * t[0] + s[1] * t[1] + s[2] * t[2] + t[RO];
  const double bc = s[RO] * dot + E * tE + s[bt1] * t[bt1] + s[bt2] * t[bt2];
  bE += c * tE;
  bpt += t[vn] + s[vn] * tE;
  bvB -= s[bn] * tE;
  double bro = c * dot, bp = bpt + r1 * bE, bB2 = 0.5 * (bpt + bE);
  double bv[3] = {0, 0, 0}, bB[3] = {0, 0, 0};
  bv[vn] = bc + rc * t[vn] + pt * tE;
  bv[vt1] = rc * t[vt1] - s[bn] * t[bt1];
  bv[vt2] = rc * t[vt2] - s[bn] * t[bt2];
  bB[vn] = -(2 * s[bn] * t[vn] + s[bt1] * t[vt1] + s[bt2] * t[vt2] + s[vt1] * t[bt1] + s[vt2] * t[bt2] + vB * tE);
  bB[vt1] = c * t[bt1] - s[bn] * t[vt1];
  bB[vt2] = c * t[bt2] - s[bn] * t[vt2];
  // af = (A + sqrt(max(q, 0))) / (2 ro), A = f1 + B2, q = A*A - f1*f2
  {
    const double B2 = s[5] * s[5] + s[6] * s[6] + s[7] * s[7];
    const double f1 = kGam * s[PR], f2 = 4 * (s[bn] * s[bn]), A = f1 + B2;
    const double q = A * A - f1 * f2;
    const double sq = root(q > 0 ? q : 0.0), ir = rinv(s[RO]), bN = 0.5 * ba * ir;
    bro -= ba * af * ir;
    const double bq = (q > 0 && sq > 0) ? bN * 0.5 * rinv(sq) : 0.0;
    const double bA = bN + 2 * A * bq;
    bp += kGam * (bA - f2 * bq);
    bB2 += bA;
    bB[vn] -= 8 * s[bn] * (f1 * bq);
  }
  // E = 0.5 (ro v2 + B2) + r1 p, pt = p + 0.5 B2, vB = v . B
  const double v2 = s[0] * s[0] + s[1] * s[1] + s[2] * s[2], rE = s[RO] * bE;
  bs[RO] += bro + 0.5 * v2 * bE;
  bs[PR] += bp;
  for (int m = 0; m < 3; m++) {
    bs[m] += bv[m] + s[5 + m] * bvB + s[m] * rE;
    bs[5 + m] += bB[m] + s[m] * bvB + 2 * s[5 + m] * bB2;
  }
}

// the reverse of roS enS = Q / (aS - aM), the star energy of HLLD and HLLC-G:
// Q = (aS - vn) E - ptS vn + pt aM + Uh[bn] P, P = vB - aM Uh[bn] - w1 c1 - w2 c2,
// given bQ; w and c are the transverse velocity and field that P is formed with
#define OMHD_STAR_ENERGY(S, aS, ES, ptS, enS, P, bQ, w1, w2, c1, c2, bw1, bw2, bc1, bc2, baS, bES, bptS, bvBS, bS) \
  do {                                                                                                            \
    const double bd_ = -(bQ) * (enS);                                                                             \
    baS += bd_ + (ES) * (bQ);                                                                                     \
    bS[vn] -= ((ES) + (ptS)) * (bQ);                                                                              \
    bES += ((aS) - S[vn]) * (bQ);                                                                                 \
    bptS -= S[vn] * (bQ);                                                                                         \
    bpt += aM * (bQ);                                                                                             \
    const double bP_ = Ubn * (bQ);                                                                                \
    baM += pt * (bQ) - bd_ - Ubn * bP_;                                                                           \
    bUh[bn] += (P) * (bQ)-aM * bP_;                                                                               \
    bvBS += bP_;                                                                                                  \
    bw1 -= (c1) * bP_;                                                                                            \
    bc1 -= (w1) * bP_;                                                                                            \
    bw2 -= (c2) * bP_;                                                                                            \
    bc2 -= (w2) * bP_;                                                                                            \
  } while (0)

// bL += (dF/dL)^T bF, bR += (dF/dR)^T bF at the branch hlld_fwd takes.
template <int D>
OMHD_HD void hlld_vjp(const double L[NV], const double R[NV], double ch, const double bF[NV], double bL[NV],
                      double bR[NV]) {
  constexpr int vn = D, vt1 = (D + 1) % 3, vt2 = (D + 2) % 3;
  constexpr int mn = vn, mt1 = vt1, mt2 = vt2;
  constexpr int bn = 5 + vn, bt1 = 5 + vt1, bt2 = 5 + vt2;
  constexpr int RO = 4, EN = 3, PS = 8;
  const double hllg = 1.001;
  double EL, ER, ptL, ptR, vBL, vBR, afL, afR, sa, aL, aR;
  double Uh[NV];  // slots mn, mt1, mt2, RO, bn, bt1, bt2
  // the two sides' terms t, and the fan speed e of FS - e US
  double tL[NV], tR[NV], eL = 0, eR = 0;
  double baL = 0, baR = 0, bptL = 0, bptR = 0, bvBL = 0, bvBR = 0, bEL = 0, bER = 0;
  {
    SideFwd<D> l, r;
    side_fwd<D>(L, l);
    side_fwd<D>(R, r);
    EL = l.E, ptL = l.pt, vBL = l.vB, afL = l.af;
    ER = r.E, ptR = r.pt, vBR = r.vB, afR = r.af;
    sa = root(tmax(afL, afR));
    aL = tmin(L[vn], R[vn]) - sa;
    aR = tmax(L[vn], R[vn]) + sa;
    const double iw = 1.0 / (aR - aL);
    for (int m = 0; m < 3; m++) Uh[m] = iw * (aR * (R[RO] * R[m]) - aL * (L[RO] * L[m]) - r.F[m] + l.F[m]);
    for (int m = RO; m <= 7; m++) Uh[m] = iw * (aR * R[m] - aL * L[m] - r.F[m] + l.F[m]);
  }
  {  // GLM pair (flux_solver.f90:580-581), every branch
    OMHD_CONTRACT
    bL[PS] += 0.5 * bF[bn] + 0.5 * ch * bF[PS];
    bR[PS] += 0.5 * bF[bn] - 0.5 * ch * bF[PS];
    bL[bn] += 0.5 * ch * bF[bn] + 0.5 * ch * ch * bF[PS];
    bR[bn] += -0.5 * ch * bF[bn] + 0.5 * ch * ch * bF[PS];
  }
  tL[bn] = tR[bn] = tL[PS] = tR[PS] = 0.0;
  if (aL >= 0 || aR <= 0) {
    const double kL = aL >= 0 ? 1.0 : 0.0, kR = aL >= 0 ? 0.0 : 1.0;
    for (int m = 0; m < 8; m++)
      if (m != bn) {
        tL[m] = kL * bF[m];
        tR[m] = kR * bF[m];
      }
  } else {
    const double aM = Uh[mn] / Uh[RO];
    const double roL = L[RO] * (aL - L[vn]) / (aL - aM);
    const double roR = R[RO] * (aR - R[vn]) / (aR - aM);
    const double Ubn = Uh[bn], hb = tabs(Ubn);
    const double sroL = root(roL), sroR = root(roR);
    const double aVL = hb / sroL;
    const double aVR = hb / sroR;
    const bool hllc = (aL >= (aM - hllg * aVL)) || ((aM + hllg * aVR) >= aR);
    const double aL1 = aM - aVL;
    const double aR1 = aM + aVR;
    {
    OMHD_CONTRACT
    const double iw = rinv(aR - aL), iro = rinv(Uh[RO]), idL = rinv(aL - aM), idR = rinv(aR - aM);
    const double dL = aL - L[vn], dR = aR - R[vn];
    const double pt = ptL + L[RO] * dL * (aM - L[vn]);
    double bUh[NV] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    double baM = 0, bpt = 0, broL = 0, broR = 0;
    eL = aL;
    eR = aR;
    tL[EN] = tR[EN] = 0.0;
    if (hllc) {
      // ---- HLLC-G (flux_solver.f90:447-476) ----
      const double at1 = Uh[mt1] * iro, at2 = Uh[mt2] * iro;
      double bat1 = 0, bat2 = 0;
      auto side = [&](const double *S, double *bS, double *tS, const double aS, const double idS, const double roS,
                      const double ES, const double ptS, const double vBS, double &baS, double &broS, double &bES,
                      double &bptS, double &bvBS) __attribute__((always_inline)) {
        OMHD_CONTRACT
        const double P = vBS - aM * Ubn - at1 * Uh[bt1] - at2 * Uh[bt2];
        const double enS = ((aS - S[vn]) * ES - ptS * S[vn] + pt * aM + Ubn * P) * idS;
        const double row = bF[RO] + aM * bF[mn] + at1 * bF[mt1] + at2 * bF[mt2];
        const double x = aS * roS, bQ = aS * bF[EN] * idS;
        tS[mn] = bF[mn];
        tS[mt1] = bF[mt1];
        tS[mt2] = bF[mt2];
        tS[RO] = bF[RO];
        tS[EN] = bF[EN];
        baS += roS * row + enS * bF[EN];
        broS += aS * row;
        baM += x * bF[mn];
        bat1 += x * bF[mt1];
        bat2 += x * bF[mt2];
        OMHD_STAR_ENERGY(S, aS, ES, ptS, enS, P, bQ, at1, at2, Uh[bt1], Uh[bt2], bat1, bat2, bUh[bt1], bUh[bt2], baS,
                         bES, bptS, bvBS, bS);
      };
      tL[mn] = tL[mt1] = tL[mt2] = tL[RO] = tR[mn] = tR[mt1] = tR[mt2] = tR[RO] = 0.0;
      // s1 = 0.5 + SIGN(0.5, aM) is 1 (left) or 0
      if (csign(0.5, aM) > 0) side(L, bL, tL, aL, idL, roL, EL, ptL, vBL, baL, broL, bEL, bptL, bvBL);
      else side(R, bR, tR, aR, idR, roR, ER, ptR, vBR, baR, broR, bER, bptR, bvBR);
      bUh[mt1] += bat1 * iro;
      bUh[mt2] += bat2 * iro;
      bUh[RO] -= (at1 * bat1 + at2 * bat2) * iro;
      // F[bt] = iw (aR FL - aL FR + aL aR (R - L)): FL - aL L with the factor iw aR, FR - aR R with -iw aL
      double g = 0;
      for (int q = 0; q < 2; q++) {
        const int bt = q ? bt2 : bt1, vt = q ? vt2 : vt1;
        const double be = iw * bF[bt];
        const double fl = L[vn] * L[bt] - L[bn] * L[vt], fr = R[vn] * R[bt] - R[bn] * R[vt];
        tL[bt] = aR * be;
        tR[bt] = -aL * be;
        baL += (aR * R[bt] - fr) * be;
        baR += (fl - aL * L[bt]) * be;
        g += iw * (aR * fl - aL * fr + aL * aR * (R[bt] - L[bt])) * be;
      }
      baR -= g;
      baL += g;
    } else {
      // ---- HLLD (flux_solver.f90:482-572) ----
      const double f1L = rinv(L[RO] * dL * (aL - aM) - Ubn * Ubn), f1R = rinv(R[RO] * dR * (aR - aM) - Ubn * Ubn);
      const double gL = f1L * (L[RO] * dL * dL - Ubn * Ubn), gR = f1R * (R[RO] * dR * dR - Ubn * Ubn);
      const double b1L = L[bt1] * gL, b2L = L[bt2] * gL, b1R = R[bt1] * gR, b2R = R[bt2] * gR;
      const double hL = f1L * Ubn * (aM - L[vn]), hR = f1R * Ubn * (aM - R[vn]);
      const double v1L = L[vt1] - hL * L[bt1], v2L = L[vt2] - hL * L[bt2];
      const double v1R = R[vt1] - hR * R[bt1], v2R = R[vt2] - hR * R[bt2];
      const bool central = aL1 < 0 && aR1 > 0;
      const bool left = central ? aM >= 0 : aL1 >= 0;
      const double kL = left ? 1.0 : 0.0, kR = left ? 0.0 : 1.0;
      const double isL = rinv(sroL), isR = rinv(sroR);
      double bv1L = 0, bv2L = 0, bv1R = 0, bv2R = 0, bb1L = 0, bb2L = 0, bb1R = 0, bb2R = 0;
      double bsL = 0, bsR = 0, ba1L = 0, ba1R = 0;  // sqrt(roS), aL1 and aR1
      if (central) {  // central states (flux_solver.f90:533-572)
        const double sB = csign(1.0, Ubn), fc = rinv(sroL + sroR), P = sroL * sroR * sB;
        const double at1 = fc * (sroL * v1L + sroR * v1R + (b1R - b1L) * sB);
        const double at2 = fc * (sroL * v2L + sroR * v2R + (b2R - b2L) * sB);
        const double B1 = fc * (sroL * b1R + sroR * b1L + P * (v1R - v1L));
        const double B2 = fc * (sroL * b2R + sroR * b2L + P * (v2R - v2L));
        // the side taken: U2 = (roT, roT aM, roT at, UT1[EN] + sT K, B)
        const double w = left ? aL1 : aR1, roT = left ? roL : roR, sT = left ? -sroL * sB : sroR * sB;
        const double v1T = left ? v1L : v1R, v2T = left ? v2L : v2R, b1T = left ? b1L : b1R, b2T = left ? b2L : b2R;
        const double K = v1T * b1T + v2T * b2T - at1 * B1 - at2 * B2;
        const double bK = w * bF[EN] * sT, wr = w * roT, bs = K * sB * w * bF[EN];
        const double ba1 = roT * ((at1 - v1T) * bF[mt1] + (at2 - v2T) * bF[mt2]) + sT * K * bF[EN] +
                           (B1 - b1T) * bF[bt1] + (B2 - b2T) * bF[bt2];
        const double bro = w * (at1 * bF[mt1] + at2 * bF[mt2]);
        ba1L = kL * ba1;
        ba1R = kR * ba1;
        broL += kL * bro;
        broR += kR * bro;
        // fc (at), fc (B) reversed: a = fc bat, n = fc bB
        const double a1 = fc * (wr * bF[mt1] - B1 * bK), a2 = fc * (wr * bF[mt2] - B2 * bK);
        const double n1 = fc * (w * bF[bt1] - at1 * bK), n2 = fc * (w * bF[bt2] - at2 * bK);
        const double z = at1 * a1 + at2 * a2 + B1 * n1 + B2 * n2;  // the adjoint of fc times -fc
        const double bP = ((v1R - v1L) * n1 + (v2R - v2L) * n2) * sB;
        bsL = b1R * n1 + b2R * n2 + v1L * a1 + v2L * a2 + sroR * bP - z - kL * bs;
        bsR = b1L * n1 + b2L * n2 + v1R * a1 + v2R * a2 + sroL * bP - z + kR * bs;
        const double KL = kL * bK, KR = kR * bK;
        bv1L = sroL * a1 - P * n1 + KL * b1L;
        bv2L = sroL * a2 - P * n2 + KL * b2L;
        bv1R = sroR * a1 + P * n1 + KR * b1R;
        bv2R = sroR * a2 + P * n2 + KR * b2R;
        bb1L = sroR * n1 - sB * a1 + KL * v1L;
        bb2L = sroR * n2 - sB * a2 + KL * v2L;
        bb1R = sroL * n1 + sB * a1 + KR * v1R;
        bb2R = sroL * n2 + sB * a2 + KR * v2R;
      }
      // aL1 = aM - aVL, aR1 = aM + aVR, aVS = |Uh[bn]| / sqrt(roS)
      baM += ba1L + ba1R;
      bUh[bn] += (Ubn < 0 ? -1.0 : 1.0) * (ba1R * isR - ba1L * isL);
      broL += 0.5 * isL * (bsL + ba1L * aVL * isL);
      broR += 0.5 * isR * (bsR - ba1R * aVR * isR);
      // the star states, reversed side by side
      auto star = [&](const double *S, double *bS, double *tS, const double k, const double aS, const double y,
                      const double dS, const double idS, const double roS, const double ES, const double ptS,
                      const double vBS, const double f1, const double g, const double v1, const double v2,
                      const double b1, const double b2, double bv1, double bv2, double bb1, double bb2, double &baS,
                      double &broS, double &bES, double &bptS, double &bvBS) __attribute__((always_inline)) {
        OMHD_CONTRACT
        // F takes aS US1 (S*), or (aS - aS1) US1 + aS1 U2 (S**): y is the factor of US1's transverse parts
        const double P = vBS - aM * Ubn - v1 * b1 - v2 * b2;
        const double en = (dS * ES - ptS * S[vn] + pt * aM + Ubn * P) * idS;
        const double x = k * aS, row = bF[RO] + aM * bF[mn], rot = v1 * bF[mt1] + v2 * bF[mt2];
        for (int m = 0; m < 8; m++)
          if (m != bn) tS[m] = k * bF[m];
        baS += k * (roS * (row + rot) + en * bF[EN] + b1 * bF[bt1] + b2 * bF[bt2]);
        broS += x * row + y * rot;
        baM += x * roS * bF[mn];
        bv1 += y * roS * bF[mt1];
        bv2 += y * roS * bF[mt2];
        bb1 += y * bF[bt1];
        bb2 += y * bF[bt2];
        const double bQ = x * bF[EN] * idS;
        OMHD_STAR_ENERGY(S, aS, ES, ptS, en, P, bQ, v1, v2, b1, b2, bv1, bv2, bb1, bb2, baS, bES, bptS, bvBS, bS);
        // v = S[vt] - f1 Uh[bn] S[bt] (aM - vn), b = S[bt] f1 e, e = ro (aS - vn)^2 - Uh[bn]^2,
        // 1/f1 = ro (aS - vn) (aS - aM) - Uh[bn]^2
        const double c = aM - S[vn], fU = f1 * Ubn;
        const double sv = S[bt1] * bv1 + S[bt2] * bv2, sb = S[bt1] * bb1 + S[bt2] * bb2;
        bS[vt1] += bv1;
        bS[vt2] += bv2;
        bS[bt1] += g * bb1 - fU * c * bv1;
        bS[bt2] += g * bb2 - fU * c * bv2;
        const double be = f1 * sb, bd = -f1 * (g * sb - fU * c * sv), p2 = aS - aM, rd = S[RO] * dS, rp = S[RO] * p2;
        baM -= fU * sv + rd * bd;
        bUh[bn] -= f1 * c * sv + 2 * Ubn * (be + bd);
        bS[RO] += dS * (dS * be + p2 * bd);
        baS += 2 * rd * be + (rp + rd) * bd;
        bS[vn] += fU * sv - 2 * rd * be - rp * bd;
      };
      star(R, bR, tR, kR, aR, kR * (central ? aR - aR1 : aR), dR, idR, roR, ER, ptR, vBR, f1R, gR, v1R, v2R, b1R, b2R,
           bv1R, bv2R, bb1R, bb2R, baR, broR, bER, bptR, bvBR);
      star(L, bL, tL, kL, aL, kL * (central ? aL - aL1 : aL), dL, idL, roL, EL, ptL, vBL, f1L, gL, v1L, v2L, b1L, b2L,
           bv1L, bv2L, bb1L, bb2L, baL, broL, bEL, bptL, bvBL);
    }
    // roS = S[RO] (aS - vn) / (aS - aM)
    const double nL = broL * idL, nR = broR * idR;
    bL[RO] += dL * nL;
    baL += (L[RO] - roL) * nL;
    bL[vn] -= L[RO] * nL;
    bR[RO] += dR * nR;
    baR += (R[RO] - roR) * nR;
    bR[vn] -= R[RO] * nR;
    baM += roL * nL + roR * nR;
    // pt = ptL + L[RO] (aL - vn) (aM - vn)
    {
      const double c = aM - L[vn], bc1 = c * bpt, bc2 = L[RO] * dL * bpt;
      bptL += bpt;
      bL[RO] += dL * bc1;
      baL += L[RO] * bc1;
      bL[vn] -= L[RO] * bc1 + bc2;
      baM += bc2;
    }
    // aM = Uh[mn] / Uh[RO]
    bUh[mn] += baM * iro;
    bUh[RO] -= baM * aM * iro;
    // Uh = iw (aR UR - aL UL - FR + FL), iw = 1 / (aR - aL)
    double g = 0;
    for (int m = 0; m < 8; m++) {
      if (m == EN) continue;
      const double b = iw * bUh[m];
      g += Uh[m] * b;
      if (m == bn) {
        bR[bn] += aR * b;
        bL[bn] -= aL * b;
        baR += R[bn] * b;
        baL -= L[bn] * b;
      } else {
        tL[m] += b;
        tR[m] -= b;
      }
    }
    baL += g - (L[RO] * (L[0] * tL[0] + L[1] * tL[1] + L[2] * tL[2]) + EL * tL[EN] + L[RO] * tL[RO] +
                L[bt1] * tL[bt1] + L[bt2] * tL[bt2]);
    baR -= g + (R[RO] * (R[0] * tR[0] + R[1] * tR[1] + R[2] * tR[2]) + ER * tR[EN] + R[RO] * tR[RO] +
                R[bt1] * tR[bt1] + R[bt2] * tR[bt2]);
    }
  }
  // fan speeds: aL = min(vnL, vnR) - sa, aR = max(vnL, vnR) + sa, sa = sqrt(max(afL, afR))
  if (L[vn] < R[vn]) bL[vn] += baL;
  else bR[vn] += baL;
  if (L[vn] > R[vn]) bL[vn] += baR;
  else bR[vn] += baR;
  const double bm = (baR - baL) * (0.5 * rinv(sa));
  side_vjp<D>(L, tL, eL, EL, ptL, vBL, afL, afL > afR ? bm : 0.0, bptL, bvBL, bEL, bL);
  side_vjp<D>(R, tR, eR, ER, ptR, vBR, afR, afL > afR ? 0.0 : bm, bptR, bvBR, bER, bR);
}

#undef OMHD_STAR_ENERGY
#undef OMHD_CONTRACT

}  // namespace adj
}  // namespace omhd
