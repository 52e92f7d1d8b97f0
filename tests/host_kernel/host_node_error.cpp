// Rounding errors of node_values and of the dual-number waveform (Phenom::amp_phase) against the same
// formulas in extended precision, for tests/test_host_nodes_error.py: random binaries, the setup table's
// values taken as exact, M f log-uniform between two given values (the second in units of the mode's
// cut, short of the taper).  Prints per mode the rms errors of A, dA/du, Psi and dPsi/du by both, in
// units of 2^-53 of the terms each is the sum of.
#include <hip/hip_runtime.h>  // the host stand-in (tests/host_kernel/stub)

#include <cmath>
#include <cstdio>
#include <cstdlib>

namespace pes {  // before dual.hpp, whose templates take them for long double
inline long double dsqrt(long double x) { return std::sqrt(x); }
inline long double dlog(long double x) { return std::log(x); }
inline long double dexp(long double x) { return std::exp(x); }
inline long double datan(long double x) { return std::atan(x); }
inline long double dpow(long double x, double p) {
  return p == -7.0 / 6.0 ? 1.0L / (x * std::sqrt(std::cbrt(x))) : std::pow(x, (long double)p);
}
inline long double dcbrt(long double x) { return std::cbrt(x); }
inline long double dsin(long double x) { return std::sin(x); }
inline long double dcos(long double x) { return std::cos(x); }
}  // namespace pes

#include "phenom.hpp"

using namespace pes;

typedef Dual<long double, 1> Q;
struct TableValues {  // a row of the setup table as constants
  const double* su;
  Q operator[](int i) const { return lift<Q>(su[i]); }
};

int main(int argc, char** argv) {
  std::srand(argc > 1 ? std::atoi(argv[1]) : 1);
  const double x_lo = argc > 2 ? std::atof(argv[2]) : 2e-4, x_hi = argc > 3 ? std::atof(argv[3]) : 0.9;
  auto U = [](double a, double b) { return a + (b - a) * (std::rand() / (double)RAND_MAX); };
  typedef Dual<double, 4> D4;
  typedef Dual<Dual<double, 1>, 4> S;
  static Phenom<D4> ph;
  static double su[N_SETUP * 5];
  double sq[6][2][4] = {};
  long count[6] = {};
  for (int it = 0; it < 600; ++it) {
    D4 in[4] = {lift<D4>(std::exp(U(std::log(1e4), std::log(5e6)))), lift<D4>(U(0.1, 1.0)), lift<D4>(U(-0.9, 0.9)),
                lift<D4>(U(-0.9, 0.9))};
    for (int k = 0; k < 4; ++k) in[k].d[k] = 1.0;
    phenom_setup(ph, in[0], in[1], in[2], in[3], 0.0);
    for (int i = 0; i < N_SETUP; ++i) {
      su[i] = ph.c[i].v;
      for (int k = 0; k < 4; ++k) su[(1 + k) * N_SETUP + i] = ph.c[i].d[k];
    }
    Phenom<S, SetupView<S>> dual{SetupView<S>{su}};
    Phenom<Q, TableValues> exact{TableValues{su}};
    for (int mode = 0; mode < 6; ++mode) {
      const double m = kModeM[mode], rho = su[SU_FRD] / su[su_frd(mode)], cut = mode == 0 ? MF_CUT : MF_CUT / rho;
      for (int j = 0; j < 40; ++j) {
        const double f = std::exp(U(std::log(x_lo), std::log(x_hi * cut))) / su[SU_MSEC];
        const FreqPow q = freq_pow(f);
        Q xq = lift<Q>(f), Aq, Pq;
        xq.v *= (long double)su[SU_MSEC];
        xq.d[0] = xq.v;
        exact.amp_phase(mode, xq, Aq, Pq);
        S x = lift<S>(f * su[SU_MSEC]), A, P;
        x.v.d[0] = x.v.v;
        for (int k = 0; k < 4; ++k) x.d[k].v = x.d[k].d[0] = f * su[(1 + k) * N_SETUP + SU_MSEC];
        dual.amp_phase(mode, x, A, P);
        double v[4];
        node_values(su, mode, q, v[0], v[1], v[2], v[3]);
        const double w[4] = {A.v.v, A.v.d[0], P.v.v, P.v.d[0]};
        const long double r[4] = {Aq.v, Aq.d[0], Pq.v, Pq.d[0]};
        const double t0 = std::fabs(su[SU_T0]) * (double)xq.v, ph0 = 0.5 * m * (std::fabs(su[SU_PHIREF0]) + t0);
        double a = std::fabs((double)r[0]);
        if (mode == 1) {  // a difference: the sum of its terms
          const Q y = exact.fmap(mode, xq);
          const double v = std::cbrt(PI * (double)y.v);
          a = std::fabs((double)exact.amplitude(y).v * su[SU_AMPSCALE]) * std::sqrt(2.0) / 3.0 *
              (su[SU_DELTA] * v + 1.5 * std::fabs(su[SU_CHIA] + su[SU_DELTA] * su[SU_CHIS]) * v * v);
        }
        const double s[4] = {a, a, std::fabs((double)r[2]) + ph0,
                             std::fabs((double)r[3]) + 0.5 * m * t0};
        for (int i = 0; i < 4; ++i) {
          const double e = (double)(v[i] - r[i]) / s[i], d = (double)(w[i] - r[i]) / s[i];
          sq[mode][0][i] += e * e;
          sq[mode][1][i] += d * d;
        }
        ++count[mode];
      }
    }
  }
  for (int mode = 0; mode < 6; ++mode) {
    for (int i = 0; i < 4; ++i)
      std::printf("%.4f %.4f  ", std::sqrt(sq[mode][0][i] / count[mode]) * 0x1p53,
                  std::sqrt(sq[mode][1][i] / count[mode]) * 0x1p53);
    std::printf("\n");
  }
  return 0;
}
