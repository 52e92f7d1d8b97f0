// Host build of node_values and node_adjoint against the dual-number waveform Phenom::amp_phase, for
// tests/test_host_nodes.py: random binaries, every mode, M f from 5e-5 to beyond every cut and at
// both sides of every region's edge.  Prints the largest errors of A, dA/du, Psi, dPsi/du, each in
// units of the terms that it is the sum of, and of the gradients of A, Psi and dPsi/du, in units of
// their norms over the parameters (Psi and dPsi/du together: each passes through zero).
#include <hip/hip_runtime.h>  // the host stand-in (tests/host_kernel/stub)

#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "phenom.hpp"

using namespace pes;

int main(int argc, char** argv) {
  std::srand(argc > 1 ? std::atoi(argv[1]) : 1);
  auto U = [](double a, double b) { return a + (b - a) * (std::rand() / (double)RAND_MAX); };
  typedef Dual<double, 4> D4;
  typedef Dual<Dual<double, 1>, 4> S;
  double worst[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  static Phenom<D4> ph;
  static double su[N_SETUP * 5];
  for (int it = 0; it < 300; ++it) {
    D4 in[4] = {lift<D4>(std::exp(U(std::log(2e5), std::log(5e6)))), lift<D4>(it % 20 == 0 ? 1.0 : U(0.1, 1.0)),
                lift<D4>(U(-0.9, 0.9)), lift<D4>(U(-0.9, 0.9))};
    for (int k = 0; k < 4; ++k) in[k].d[k] = 1.0;
    phenom_setup(ph, in[0], in[1], in[2], in[3], 0.0);
    for (int i = 0; i < N_SETUP; ++i) {
      su[i] = ph.c[i].v;
      for (int k = 0; k < 4; ++k) su[(1 + k) * N_SETUP + i] = ph.c[i].d[k];
    }
    Phenom<S, SetupView<S>> ref{SetupView<S>{su}};
    for (int mode = 0; mode < 6; ++mode) {
      const double m = kModeM[mode], fi = 0.5 * m * HM_MAP_JOIN, fr = su[su_frd(mode)], rho = su[SU_FRD] / fr;
      const double cut = mode == 0 ? MF_CUT : MF_CUT / rho;
      const double edges[] = {0.5 * m * AMP_F_INS, 0.5 * m * PHI_F_INS, fi, fr, su[SU_FMAX] / rho, 0.5 * su[SU_FRD] / rho,
                              (1.0 - TAPER) * cut, cut};
      for (int j = 0; j < 60; ++j) {
        const double x = j < 16 ? edges[j / 2] * (j % 2 ? 1.0 + 1e-9 : 1.0 - 1e-9)
                                : std::exp(U(std::log(5e-5), std::log(1.05 * cut)));
        const double f = x / su[SU_MSEC], c = std::cbrt(f);
        const FreqPow q = {f, c, 1.0 / c, std::log(f), std::pow(f, -7.0 / 6.0)};
        S Mf = lift<S>(f * su[SU_MSEC]), A, P;
        Mf.v.d[0] = Mf.v.v;
        for (int k = 0; k < 4; ++k) Mf.d[k].v = Mf.d[k].d[0] = f * su[(1 + k) * N_SETUP + SU_MSEC];
        ref.amp_phase(mode, Mf, A, P);
        double v[4];
        node_values(su, mode, q, v[0], v[1], v[2], v[3]);
        const double r[4] = {A.v.v, A.v.d[0], P.v.v, P.v.d[0]}, hm = 0.5 * m;
        const NodeY n = node_y(su, mode, q);
        double phi, G;
        node_phi(su, n.y, n.c, n.ic, n.l, phi, G);
        const double st = std::fabs(su[SU_T0]) * (n.y + su[SU_MFREF]);
        // the amplitude before the taper (which itself goes to zero)
        const double a0 = std::fabs(su[SU_PRE] * n.y76) * (mode == 0 ? 1.0 : 0.02);
        const double scale[4] = {a0, a0, hm * (std::fabs(phi) + std::fabs(su[SU_PHIREF0]) + st),
                                 hm * n.r * (std::fabs(G) + st)};
        for (int i = 0; i < 4; ++i) worst[i] = std::fmax(worst[i], std::fabs(v[i] - r[i]) / scale[i]);
        double g[3][4] = {}, e[3] = {0.0, 0.0, 0.0}, nrm[3] = {0.0, 0.0, 0.0};
        for (int o = 0; o < 3; ++o) node_adjoint(su, mode, q, o == 0, o == 1, o == 2, g[o]);
        for (int k = 0; k < 4; ++k) {
          const double th = k == 0 ? in[0].v : 1.0, d[3] = {A.d[k].v, P.d[k].v, P.d[k].d[0]};
          for (int o = 0; o < 3; ++o) {
            e[o] += std::fabs(g[o][k] - d[o]) * th;
            nrm[o] += std::fabs(d[o]) * th;
          }
        }
        // the amplitude's gradient in units of the untapered amplitude's size where that is larger
        worst[4] = std::fmax(worst[4], e[0] / (nrm[0] + a0));
        worst[5] = std::fmax(worst[5], std::fmax(e[1], e[2]) / (nrm[1] + nrm[2]));
      }
    }
  }
  for (double w : worst) std::printf("%.3e ", w);
  std::printf("\n");
  return 0;
}
