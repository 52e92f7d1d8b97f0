// A, dA/du, Psi, dPsi/du (u = ln f) of one mode at one frequency from a row of the setup table, and
// the adjoint of A, Psi and dPsi/du.
//
// Every ansatz of the waveform but the ringdown's is a sum of powers of y = f22 and ln y, so y d/dy
// of a term is a multiple of the term: values and slopes come from the same powers.  The powers of y
// are products of those of f, which are the same for all rows and tabulated per node or bin, and of
// those of the mass in seconds, which are constants of the row: no cube root, logarithm or power is
// taken per (row, frequency) outside a higher mode's merger.  One Newton step from y itself takes the
// products' roundings out again (y_powers): without it A and Psi were 1.5 times further from
// extended precision than with the functions taken per frequency (tests/test_host_nodes_error.py).
// su: the row's setup table [5][N_SETUP].
#pragma once

namespace pes {

// a frequency: f, f^(1/3), f^(-1/3), ln f, f^(-7/6); the table of n frequencies is [N_FPOW][n]
constexpr int N_FPOW = 5;
struct FreqPow {
  double f, c, ic, l, f76;
};
PES_HD FreqPow load_fpow(const double* t, size_t n, size_t i) {
  return {t[i], t[n + i], t[2 * n + i], t[3 * n + i], t[4 * n + i]};
}
PES_HD FreqPow freq_pow(double f) {
  const double c = cbrt(f), ic = 1.0 / c;
  return {f, c, ic, log(f), ic * ic * ic * sqrt(ic)};
}

struct NodeY {
  double x, y, r;          // M f, f22, d ln y / d ln x
  double c, ic, l, y76;    // y^(1/3), y^(-1/3), ln y, y^(-7/6)
};
// y^(1/3), y^(-1/3) and y^(-7/6) of y from i = y^(-1/3) and p = y^(-7/6) to a few roundings: the residual
// t = 1 - y i^3, formed with the products' rounding errors, corrects all of them
PES_HD void y_powers(double y, double i, double p, NodeY& o) {
  const double i2 = i * i, e2 = fma(i, i, -i2);
  const double i3 = i2 * i, e3 = fma(e2, i, fma(i2, i, -i3));
  const double t = fma(-y, e3, fma(-y, i3, 1.0)), t3 = t * (1.0 / 3.0);
  const double h = y * i2;
  o.ic = fma(i, t3, i);
  o.c = h + (fma(y, i2, -h) + fma(y, e2, (2.0 * h) * t3));
  const double s = p * y;  // y^(-1/6), corrected by its square
  o.y76 = fma(i3, t, i3) * fma(0.5 * s * o.c, fma(-s, s, o.ic), s);
}
PES_HD int su_frd(int mode) {
  return mode == 1 ? SU_FRD21 : mode == 2 ? SU_FRD33 : mode == 3 ? SU_FRD32 : mode == 4 ? SU_FRD44
         : mode == 5 ? SU_FRD43 : SU_FRD;
}
// (2 / m)^(-1/3), ln(2 / m), (2 / m)^(-7/6), (2 pi / m)^(1/3) for m = 1, 2, 3, 4
struct ModePow {
  double ic, l, p76, pi13;
};
PES_HD ModePow mode_pow(int m) {
  switch (m) {
    case 1: return {0.79370052598409973738, 0.69314718055994530942, 0.44544935907016965237, 1.8452701486440284191};
    case 2: return {1.0, 0.0, 1.0, 1.4645918875615232630};
    case 3: return {1.1447142425533318678, -0.40546510810816438198, 1.6048697909004944263, 1.2794388617850086711};
    default: return {1.2599210498948731648, -0.69314718055994530942, 2.2449240966187459629, 1.1624473515096264756};
  }
}
PES_HD NodeY node_y(const double* su, int mode, const FreqPow& q) {
  NodeY o;
  o.x = q.f * su[SU_MSEC];
  o.r = 1.0;
  const double m = (double)kModeM[mode], fi = 0.5 * m * HM_MAP_JOIN;
  if (mode == 0 || o.x < fi) {
    double i = q.ic * su[SU_IM13], p = q.f76 * su[SU_M76];
    o.y = o.x;
    o.l = q.l + su[SU_LNM];
    if (kModeM[mode] != 2) {
      const ModePow k = mode_pow(kModeM[mode]);
      o.y *= 2.0 / m;
      i *= k.ic;
      p *= k.p76;
      o.l += k.l;
    }
    y_powers(o.y, i, p, o);
    return o;
  }
  const double fr = su[su_frd(mode)], FRD = su[SU_FRD], rho = FRD / fr;
  if (o.x >= fr) {
    o.y = rho * o.x;
  } else {
    const double w = fr - fi, iw = 1.0 / w, t = (o.x - fi) * iw;
    const double M0 = (2.0 / m) * w, M1 = rho * w;
    const double c2 = 3.0 * (FRD - HM_MAP_JOIN) - 2.0 * M0 - M1, c3 = 2.0 * (HM_MAP_JOIN - FRD) + M0 + M1;
    o.y = HM_MAP_JOIN + t * (M0 + t * (c2 + t * c3));
    o.r = o.x * iw * (M0 + t * (2.0 * c2 + 3.0 * t * c3)) / o.y;
  }
  o.c = cbrt(o.y);
  o.ic = 1.0 / o.c;
  o.l = log(o.y);
  o.y76 = sqrt(o.ic) / o.y;
  return o;
}
// v = cbrt(2 pi x / m) up to the join and saturating above it, and x dv/dx
PES_HD void node_beta_v(const double* su, int mode, const FreqPow& q, const NodeY& n, double& v, double& Dv) {
  const double m = (double)kModeM[mode];
  if (n.x < 0.5 * m * HM_MAP_JOIN) {  // 2 x / m = y
    v = fma(n.c, 1.4645918875615231, n.c * 1.0150910436435383e-16);  // pi^(1/3), and what that is rounded by
    Dv = v * (1.0 / 3.0);
  } else {
    const double k = mode_pow(kModeM[mode]).pi13, i = q.ic * su[SU_IM13] / k, X = n.x * (2.0 * PI / m);
    double vr = q.c * su[SU_M13] * k;
    vr = fma(vr * (1.0 / 3.0), (X - vr * vr * vr) * (i * i * i), vr);  // the products' roundings, as in y_powers
    const double vi = cbrt(PI * HM_MAP_JOIN), e = exp(1.0 - vr / vi);
    v = vi * (2.0 - e);
    Dv = e * vr * (1.0 / 3.0);
  }
}
// beta = k (b1 v + b2 v^2 + b3 v^3)
struct NodeBeta {
  double k, b1, b2, b3;
};
PES_HD NodeBeta node_beta(const double* su, int mode) {
  const double d = su[SU_DELTA], eta = su[SU_ETA];
  switch (mode) {
    case 1: return {sqrt(2.0) / 3.0, d, -1.5 * (su[SU_CHIA] + d * su[SU_CHIS]), 0.0};
    case 2: return {sqrt(2.0 / 3.0) * 0.75 * sqrt(15.0 / 14.0), d, 0.0, 0.0};
    case 3: return {(1.0 / 3.0) * sqrt(5.0 / 7.0), 0.0, 1.0 - 3.0 * eta, 0.0};
    case 4: return {sqrt(0.5) * (8.0 / 9.0) * sqrt(5.0 / 7.0), 0.0, 1.0 - 3.0 * eta, 0.0};
    default: return {sqrt(2.0 / 3.0) * (9.0 / (4.0 * sqrt(70.0))), 0.0, 0.0, d * (1.0 - 2.0 * eta)};
  }
}
// w, the taper over the end of the mode's range, and x dw/dx
PES_HD void node_taper(const double* su, int mode, double x, double& w, double& Dw) {
  w = 1.0;
  Dw = 0.0;
  const double num = mode == 0 ? 1.0 : su[SU_FRD], cut = mode == 0 ? MF_CUT : MF_CUT * su[su_frd(mode)];
  if (x * num > (1.0 - TAPER) * cut) {
    const double xc = x * num / cut, a = (xc - (1.0 - TAPER)) * (PI / TAPER);
    w = xc >= 1.0 ? 0.0 : 0.5 * (1.0 + cos(a));
    Dw = xc >= 1.0 ? 0.0 : -0.5 * sin(a) * (PI / TAPER) * xc;
  }
}
// reduced amplitude and y d/dy of it
PES_HD void node_red(const double* su, double y, double c, double& red, double& Dred) {
  auto k = [su](int i) { return su[i]; };
  if (y <= AMP_F_INS) {
    const double a2 = k(SU_A23), a3 = k(SU_A1), a4 = k(SU_A43), a5 = k(SU_A53), a6 = k(SU_A2), a7 = k(SU_RHO1),
                 a8 = k(SU_RHO2), a9 = k(SU_RHO3);
    const double c2 = c * c;
    red = 1.0 + c2 * (a2 + c * (a3 + c * (a4 + c * (a5 + c * (a6 + c * (a7 + c * (a8 + c * a9)))))));
    Dred = (1.0 / 3.0) * c2 *
           (2.0 * a2 +
            c * (3.0 * a3 + c * (4.0 * a4 + c * (5.0 * a5 + c * (6.0 * a6 + c * (7.0 * a7 + c * (8.0 * a8 + c * (9.0 * a9))))))));
  } else if (y >= k(SU_FMAX)) {
    const double F = k(SU_FDM) * k(SU_G3), d = y - k(SU_FRD), g = k(SU_G2) / F;
    const double den = 1.0 / (d * d + F * F);
    red = exp(-d * g) * (F * k(SU_G1)) * den;
    Dred = -y * red * (g + 2.0 * d * den);
  } else {
    // value and slope by one Horner scheme: the sums cancel, and the slope of what was computed errs less
    const double d4 = k(SU_D4), p3 = fma(d4, y, k(SU_D3)), p2 = fma(p3, y, k(SU_D2)), p1 = fma(p2, y, k(SU_D1));
    red = fma(p1, y, k(SU_D0));
    Dred = y * fma(fma(fma(d4, y, p3), y, p2), y, p1);
  }
}
// phase phi(y) before the alignment, and G = y d phi / dy; l = log(y)
PES_HD void node_phi(const double* su, double y, double c, double ic, double l, double& phi, double& G) {
  auto k = [su](int i) { return su[i]; };
  const double e = k(SU_IETA);
  if (y < PHI_F_INS) {
    const double c3 = c * c * c, c2 = c * c;
    const double s1 = k(SU_S1), s2 = k(SU_S2), s3 = k(SU_S3), s4 = k(SU_S4);
    const double ps = c3 * (s1 + c * (0.75 * s2 + c * (0.6 * s3 + c * (0.5 * s4))));
    const double gs = c3 * (s1 + c * (s2 + c * (s3 + c * s4)));
    const double p0 = k(SU_P0), p2 = k(SU_P2), p3 = k(SU_P3), p4 = k(SU_P4), p5 = k(SU_P5L), p7 = k(SU_P7);
    const double q6 = k(SU_P6) + k(SU_P6L) * (l + 1.1447298858494001741), ic2 = ic * ic;
    const double t = ic * (p4 + ic * (p3 + ic * (p2 + ic2 * p0))) + p5 * l + c * q6 + c2 * p7;
    const double g = p5 - (1.0 / 3.0) * (ic * (p4 + ic * (2.0 * p3 + ic * (3.0 * p2 + ic2 * (5.0 * p0))))) +
                     c * ((1.0 / 3.0) * q6 + k(SU_P6L)) + (2.0 / 3.0) * c2 * p7;
    phi = ps * e - t;
    G = gs * e - g;
  } else if (y >= 0.5 * k(SU_FRD)) {
    const double y34 = sqrt(y * sqrt(y)), iy = 1.0 / y, u = 1.0 / k(SU_FDM);
    const double z = (y - k(SU_AL5) * k(SU_FRD)) * u;
    const double c2 = k(SU_C2MRD) * y, b1 = k(SU_AL1) * y, b2 = k(SU_AL2) * iy, b3 = k(SU_AL3) * y34;
    phi = fma(fma(k(SU_AL1), y, fma(4.0 / 3.0, b3, -b2)) + k(SU_AL4) * atan(z), e, k(SU_C1MRD) + c2);
    G = (b1 + b2 + b3 + k(SU_AL4) * (y * u) / (1.0 + z * z)) * e + c2;
  } else {
    const double iy = 1.0 / y, b3 = k(SU_B3) * (iy * iy * iy), b1 = k(SU_B1) * y, c2 = k(SU_C2INT) * y;
    // (ln y anew: in the sum of logarithms those of f and M nearly cancel here)
    phi = (b1 - (1.0 / 3.0) * b3 + k(SU_B2) * log(y)) * e + k(SU_C1INT) + c2;
    G = (b1 + b3 + k(SU_B2)) * e + c2;
  }
}

PES_HD void node_values(const double* su, int mode, const FreqPow& q, double& A, double& dA, double& P, double& dP) {
  const NodeY n = node_y(su, mode, q);
  double red, Dred, phi, G, w, Dw;
  node_red(su, n.y, n.c, red, Dred);
  const double pre = n.y76 * su[SU_PRE];
  double am = red * pre, Dam = (Dred - (7.0 / 6.0) * red) * pre * n.r;
  if (mode != 0) {
    double v, Dv;
    node_beta_v(su, mode, q, n, v, Dv);
    const NodeBeta b = node_beta(su, mode);
    const double be = b.k * (v * (b.b1 + v * (b.b2 + v * b.b3)));
    const double Dbe = b.k * (Dv * (b.b1 + v * (2.0 * b.b2 + 3.0 * v * b.b3)));
    Dam = Dam * be + am * Dbe;
    am *= be;
  }
  node_taper(su, mode, n.x, w, Dw);
  A = am * w;
  dA = Dam * w + am * Dw;
  node_phi(su, n.y, n.c, n.ic, n.l, phi, G);
  const double hm = 0.5 * (double)kModeM[mode], t0 = su[SU_T0];
  P = hm * (phi - su[SU_PHIREF0] - t0 * (n.y - su[SU_MFREF]));
  dP = hm * (G - t0 * n.y) * n.r;
}

// The adjoint of A, Psi and dPsi/du at fixed f: adds wA dA/dtheta_k + wP dPsi/dtheta_k + wD
// d(dPsi/du)/dtheta_k to g[k], k = 0 .. 3 (Mc, q, chi1, chi2).  Each coefficient's adjoint is one scalar,
// contracted at once with the coefficient's four tangents.
PES_HD void node_adjoint(const double* su, int mode, const FreqPow& fq, double wA, double wP, double wD, double g[4]) {
  auto k = [su](int i) { return su[i]; };
  auto add = [su, g](int i, double s) {
#pragma unroll
    for (int q = 0; q < 4; ++q) g[q] = fma(s, su[(1 + q) * N_SETUP + i], g[q]);
  };
  const NodeY nd = node_y(su, mode, fq);
  const double x = nd.x, y = nd.y, r = nd.r, c = nd.c, ic = nd.ic, l = nd.l;
  const double hm = 0.5 * (double)kModeM[mode], t0 = k(SU_T0), e = k(SU_IETA);
  double X = 0.0;   // adjoint of ln x
  double aF = 0.0;  // adjoint of the 22 ringdown frequency
  double aE = 0.0, aeta = 0.0;  // adjoints of 1 / eta and eta
  double Y;         // adjoint of ln y
  double ar;        // adjoint of d ln y / d ln x
  // ---- phase: Psi = hm (phi - c0 - t0 (y - mfref)), dPsi = hm (G - t0 y) r
  {
    const double ap = hm * wP, ag = hm * wD * r, as = ap + ag;
    double G, DG;  // y dphi/dy and y dG/dy
    if (y < PHI_F_INS) {
      const double ic2 = ic * ic, ic3 = ic2 * ic, c2 = c * c, c3 = c2 * c;
      const double s1 = k(SU_S1), s2 = k(SU_S2), s3 = k(SU_S3), s4 = k(SU_S4);
      const double ps = c3 * (s1 + c * (0.75 * s2 + c * (0.6 * s3 + c * (0.5 * s4))));
      const double gs = c3 * (s1 + c * (s2 + c * (s3 + c * s4)));
      const double hs = c3 * (s1 + c * ((4.0 / 3.0) * s2 + c * ((5.0 / 3.0) * s3 + c * (2.0 * s4))));
      const double p0 = k(SU_P0), p2 = k(SU_P2), p3 = k(SU_P3), p4 = k(SU_P4), p6l = k(SU_P6L), p7 = k(SU_P7);
      const double L = l + 1.1447298858494001741, q6 = k(SU_P6) + p6l * L;
      const double gt = k(SU_P5L) - (1.0 / 3.0) * (ic * (p4 + ic * (2.0 * p3 + ic * (3.0 * p2 + ic2 * (5.0 * p0))))) +
                        c * ((1.0 / 3.0) * q6 + p6l) + (2.0 / 3.0) * c2 * p7;
      const double ht = (1.0 / 9.0) * (ic * (p4 + ic * (4.0 * p3 + ic * (9.0 * p2 + ic2 * (25.0 * p0)))) + c * q6) +
                        (2.0 / 3.0) * c * p6l + (4.0 / 9.0) * c2 * p7;
      G = gs * e - gt;
      DG = hs * e - ht;
      aE += ap * ps + ag * gs;
      const double ec = e * c3;
      add(SU_S1, ec * as);
      add(SU_S2, ec * c * (0.75 * ap + ag));
      add(SU_S3, ec * c2 * (0.6 * ap + ag));
      add(SU_S4, ec * c3 * (0.5 * ap + ag));
      add(SU_P0, -ic3 * ic2 * (ap - (5.0 / 3.0) * ag));
      add(SU_P2, -ic3 * (ap - ag));
      add(SU_P3, -ic2 * (ap - (2.0 / 3.0) * ag));
      add(SU_P4, -ic * (ap - (1.0 / 3.0) * ag));
      add(SU_P5L, -(ap * l + ag));
      add(SU_P6, -c * (ap + (1.0 / 3.0) * ag));
      add(SU_P6L, -c * (ap * L + ag * ((1.0 / 3.0) * L + 1.0)));
      add(SU_P7, -c2 * (ap + (2.0 / 3.0) * ag));
    } else if (y >= 0.5 * k(SU_FRD)) {
      const double y34 = sqrt(y * sqrt(y)), iy = 1.0 / y, u = 1.0 / k(SU_FDM), FRD = k(SU_FRD);
      const double z = (y - k(SU_AL5) * FRD) * u, n = 1.0 / (1.0 + z * z), q = y * u * n, at = atan(z);
      const double b1 = k(SU_AL1) * y, b2 = k(SU_AL2) * iy, b3 = k(SU_AL3) * y34, a4 = k(SU_AL4);
      const double c2 = k(SU_C2MRD) * y;
      const double gm = b1 + b2 + b3 + a4 * q;
      G = gm * e + c2;
      DG = (b1 - b2 + 0.75 * b3 + a4 * (q - 2.0 * z * n * q * (y * u))) * e + c2;
      aE += ap * (b1 - b2 + (4.0 / 3.0) * b3 + a4 * at) + ag * gm;
      add(SU_AL1, e * y * as);
      add(SU_AL2, e * iy * (ag - ap));
      add(SU_AL3, e * y34 * ((4.0 / 3.0) * ap + ag));
      add(SU_AL4, e * (ap * at + ag * q));
      const double az = e * a4 * (ap * n - 2.0 * z * n * q * ag);  // adjoint of z
      add(SU_AL5, -az * FRD * u);
      aF -= az * k(SU_AL5) * u;
      add(SU_FDM, -u * (az * z + e * a4 * ag * q));
      add(SU_C1MRD, ap);
      add(SU_C2MRD, y * as);
    } else {
      const double iy = 1.0 / y, iy3 = iy * iy * iy, b1 = k(SU_B1) * y, b3 = k(SU_B3) * iy3;
      const double c2 = k(SU_C2INT) * y;
      G = (b1 + b3 + k(SU_B2)) * e + c2;
      DG = (b1 - 3.0 * b3) * e + c2;
      aE += ap * (b1 - (1.0 / 3.0) * b3 + k(SU_B2) * l) + ag * (b1 + b3 + k(SU_B2));
      add(SU_B1, e * y * as);
      add(SU_B3, e * iy3 * (ag - (1.0 / 3.0) * ap));
      add(SU_B2, e * (ap * l + ag));
      add(SU_C1INT, ap);
      add(SU_C2INT, y * as);
    }
    add(SU_PHIREF0, -ap);
    add(SU_T0, -ap * (y - k(SU_MFREF)) - ag * y);
    add(SU_MFREF, ap * t0);
    Y = ap * (G - t0 * y) + ag * (DG - t0 * y);
    ar = hm * wD * (G - t0 * y);
  }
  // ---- amplitude: A = beta red(y) pre y^(-7/6) w
  {
    double w, Dw, be = 1.0, red, Dred;
    node_taper(su, mode, x, w, Dw);
    node_red(su, y, c, red, Dred);
    const double pre = nd.y76 * k(SU_PRE), am = red * pre;
    const double aS = wA * w;  // adjoint of beta am
    if (mode != 0) {
      double v, Dv;
      node_beta_v(su, mode, fq, nd, v, Dv);
      const NodeBeta b = node_beta(su, mode);
      be = b.k * (v * (b.b1 + v * (b.b2 + v * b.b3)));
      const double ab = aS * am;
      X += ab * b.k * Dv * (b.b1 + v * (2.0 * b.b2 + 3.0 * v * b.b3));
      const double d = k(SU_DELTA), eta = k(SU_ETA);
      if (mode == 1) {
        const double v2 = -sqrt(2.0) / 2.0 * v * v * ab;
        add(SU_DELTA, sqrt(2.0) / 3.0 * v * ab + v2 * k(SU_CHIS));
        add(SU_CHIA, v2);
        add(SU_CHIS, v2 * d);
      } else if (mode == 2) {
        add(SU_DELTA, sqrt(2.0 / 3.0) * 0.75 * sqrt(15.0 / 14.0) * v * ab);
      } else if (mode == 3) {
        aeta -= sqrt(5.0 / 7.0) * v * v * ab;
      } else if (mode == 4) {
        aeta -= sqrt(0.5) * (8.0 / 3.0) * sqrt(5.0 / 7.0) * v * v * ab;
      } else {
        const double v3 = sqrt(2.0 / 3.0) * (9.0 / (4.0 * sqrt(70.0))) * v * v * v * ab;
        add(SU_DELTA, v3 * (1.0 - 2.0 * eta));
        aeta -= 2.0 * v3 * d;
      }
    }
    const double aam = aS * be, ared = aam * pre;
    Y += ared * (Dred - (7.0 / 6.0) * red);
    add(SU_LNPRE, aam * am);
    if (Dw != 0.0) {  // the taper, a function of x / cut
      const double aw = wA * be * am * Dw;
      X += aw;
      if (mode != 0) {
        add(su_frd(mode), -aw / k(su_frd(mode)));
        aF += aw / k(SU_FRD);
      }
    }
    if (y <= AMP_F_INS) {
      double b = ared * c * c;
      const int id[8] = {SU_A23, SU_A1, SU_A43, SU_A53, SU_A2, SU_RHO1, SU_RHO2, SU_RHO3};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        add(id[i], b);
        b *= c;
      }
    } else if (y >= k(SU_FMAX)) {
      const double FDM = k(SU_FDM), F = FDM * k(SU_G3), d = y - k(SU_FRD), iF = 1.0 / F, g2 = k(SU_G2) * iF;
      const double den = 1.0 / (d * d + F * F), R = ared * red;
      add(SU_G1, ared * exp(-d * g2) * F * den);
      add(SU_G2, -R * d * iF);
      const double af = R * (iF + d * g2 * iF - 2.0 * F * den);
      add(SU_FDM, af * k(SU_G3));
      add(SU_G3, af * FDM);
      aF += R * (g2 + 2.0 * d * den);
    } else {
      double b = ared;
      const int id[5] = {SU_D0, SU_D1, SU_D2, SU_D3, SU_D4};
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        add(id[i], b);
        b *= y;
      }
    }
  }
  add(SU_IETA, aE);
  if (mode > 2) add(SU_ETA, aeta);
  // ---- the frequency map
  if (mode == 0) {
    X += Y;
  } else {
    const double m = (double)kModeM[mode], fi = 0.5 * m * HM_MAP_JOIN;
    const double fr = k(su_frd(mode)), FRD = k(SU_FRD);
    if (x < fi) {
      X += Y;
    } else if (x >= fr) {
      X += Y;
      aF += Y / FRD;
      add(su_frd(mode), -Y / fr);
    } else {
      const double rho = FRD / fr, w = fr - fi, iw = 1.0 / w, t = (x - fi) * iw;
      const double M0 = (2.0 / m) * w, M1 = rho * w;
      const double c2 = 3.0 * (FRD - HM_MAP_JOIN) - 2.0 * M0 - M1, c3 = 2.0 * (HM_MAP_JOIN - FRD) + M0 + M1;
      const double s = M0 + t * (2.0 * c2 + 3.0 * t * c3), iy = 1.0 / y;  // s = dy/dt; x dy/dx = x s / w = r y
      const double ay = (Y - ar * r) * iy, aD = ar * iy, as = aD * x * iw;
      const double a2 = ay * t * t + 2.0 * t * as, a3 = ay * t * t * t + 3.0 * t * t * as;
      const double at = ay * s + as * (2.0 * c2 + 6.0 * t * c3);
      const double a0 = ay * t + as - 2.0 * a2 + a3, a1 = a3 - a2;
      X += x * (aD * s * iw + at * iw);
      const double aw = -aD * s * x * iw * iw + a0 * (2.0 / m) + a1 * rho - at * t * iw;
      const double arho = a1 * w;
      aF += 3.0 * a2 - 2.0 * a3 + arho / fr;
      add(su_frd(mode), aw - arho * rho / fr);
    }
  }
  add(SU_FRD, aF);
  add(SU_LNM, X);
}

}  // namespace pes
