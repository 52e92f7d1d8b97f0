// Fused lnL (+ gradient) by panels: the smooth part of the response is a short polynomial.
//
// Over a panel (at most 256 consecutive bins of one node interval and one tile) everything in a
// mode's response but its total phase varies slowly with f: amplitude, link projections, pair
// phasors, sincs and the delay D.  With the channels' prefactors (pf, pfT of tdi_consts) and the
// t_c phasor taken out,
//   out_c(f) = P_c(f) sum_m u_m(f) T_{m,c}(f),   P_c = pf_c exp(-2 pi i f t_c),
//   u_m = exp(-i (Psi_m + 2 pi f k.x0)),
// each T_{m,c} (complex, c = 0, 1, 2) and k.x0(t_m(f)) is the quartic through its values at the
// five Chebyshev points of the panel, evaluated there by the same mode_geom / pair_eval as a bin.
// Psi is the node interval's Hermite cubic, P_c is exact at every bin.  The truncation lies below
// the rounding of the bin-by-bin evaluation: the five-point interpolation of a function that
// turns by theta over half the panel, or is a power f^-p over a relative half-width eps, errs by
// theta^5 / 1920 or (p)_5 eps^5 / 1920; the host cuts panels at eps <= 1.4e-3 and
// 4 pi L (f_hi - f_lo) <= 3e-3 (panel_cut.hpp), and k_panel_class sends a (tile, row) whose
// orbit angle turns by more than PANEL_SWING in a panel to the bin-by-bin kernel: ~3e-15 of
// the panel's largest |T| (interpolated against evaluated in FP64, three orbits, 1e-3 - 0.05 Hz).
// lnL and gradient against the bin-by-bin kernel: 3e-16 and 2e-14 of the largest in a batch of 15 rows.
//
// The gradient needs no per-bin adjoint either: with g_c = conj(2 w r_c) P_c u_m, the sums over
// the panel's bins M_{c,j} = sum g_c x^j (x in [-1, 1] the place in the panel) carry all of it.
// They go back to the five points (the transpose of the interpolation), and mode_adjoint runs
// there, with u = 1, instead of at every bin.
//
// What bounds it: FP64 VALU issue.  Per (bin, mode, row) ~62 instructions forward (19 for the
// sine and cosine of the phase, 24 for the six real quartics) and ~70 for the moments, against
// ~300 and ~850 for the bin-by-bin kernel; the points' geometry and the moments' reduction add
// about a fifth.  One-year network of LISA, Taiji and TianQin, six modes: 1024 rows with the
// gradient 336 -> 111 ms, 2048 without 223 -> 95 ms; one mode on a year of LISA data, 512 rows, 4.2
// -> 1.9 ms.  VALU busy 0.74 (two waves per SIMD: 256 registers); the rest is waits for LDS and L2.
//
// A wave takes one panel and NR rows (two for five or six modes, up to twelve for one) and needs
// no barrier inside: lanes <-> (row, mode, point) for the geometry, then, two rows at a time,
// lane = 32 h + l <-> bins l, l + 32, ... of row h (eight bins per lane and row: the mode's
// coefficients are read from LDS once per eight bins).
// This header is included inside the anonymous namespace of pespace_amd.hip.
#pragma once

constexpr int PANEL_K = 5;              // interpolation points
constexpr int PANEL_MIN_TILES = 512;    // contexts with fewer panel tiles go bin by bin
// doubles per panel: f_mid, 1 / f_half, f_half, s at its ends, -, then per point f, the Hermite
// weights hb1 .. he3 and sin, cos of pi f L (BinPre), and a pad to 16 bytes
constexpr int PAN_PT = 6, PAN_PT_D = 10, PAN_D = PAN_PT + PANEL_K * PAN_PT_D;
constexpr int PANEL_REC = 8;            // double2 per bin of the panel kernel's record
constexpr int PANEL_CF = 8 * PANEL_K;   // doubles per (row, mode): [j][6 T components, 2 pi k.x0, Psi]
constexpr int PANEL_PAIRS = 2 * (32 / PANEL_K);  // (row, mode) pairs of one geometry pass, at most
constexpr int PANEL_RED = 66;           // LDS row of the moments' reduction (padded: conflict-free 16-byte reads)

constexpr int PANEL_G = 13;  // LDS row of a point's gradient terms (odd: conflict-free)
constexpr int PANEL_ROWS = 12;  // rows per work item (a multiple of every geometry pass's 2, 4, 6, 12)

// cos(m pi / 10)
__host__ __device__ constexpr double cos_pi10(int m) {
  m %= 20;
  if (m > 10) m = 20 - m;
  constexpr double c[11] = {1.0, 0.95105651629515357212, 0.80901699437494742410, 0.58778525229247312917,
                            0.30901699437494742410, 0.0, -0.30901699437494742410, -0.58778525229247312917,
                            -0.80901699437494742410, -0.95105651629515357212, -1.0};
  return c[m];
}
// Chebyshev point k of PANEL_K on [-1, 1]
__host__ __device__ constexpr double panel_x(int k) { return cos_pi10(2 * k + 1); }
// coefficient of x^j per unit value at point k: the Chebyshev sums a_n = (2/5) sum_k v_k
// cos(n pi (2k + 1) / 10) (a_0 halved) written in powers of x
__host__ __device__ constexpr double panel_ci(int j, int k) {
  const double a0 = 0.2, a1 = 0.4 * cos_pi10(2 * k + 1), a2 = 0.4 * cos_pi10(2 * (2 * k + 1)),
               a3 = 0.4 * cos_pi10(3 * (2 * k + 1)), a4 = 0.4 * cos_pi10(4 * (2 * k + 1));
  return j == 0 ? a0 - a2 + a4 : j == 1 ? a1 - 3.0 * a3 : j == 2 ? 2.0 * a2 - 8.0 * a4 : j == 3 ? 4.0 * a3 : 8.0 * a4;
}

// rows of one geometry pass: NRh per half wave
__host__ __device__ inline int panel_rows_half(int n_modes) { return 32 / (PANEL_K * n_modes); }

// The bounds of t over s in [sa, sb] of a node interval (interval_t_range over part of it)
__device__ inline void panel_t_range(const double* __restrict__ n, double fa, double fb, double sa, double sb, double du,
                                     double tc, double& tl, double& th) {
  const double dP = n[6] - n[2], c = du * n[3], d1 = du * n[7];
  const double a = 3.0 * (c + d1) - 6.0 * dP, bq = 6.0 * dP - 4.0 * c - 2.0 * d1;
  const double va = fma(sa, fma(sa, a, bq), c), vb = fma(sb, fma(sb, a, bq), c);
  double lo = fmin(va, vb), hi = fmax(va, vb);
  if (a != 0.0) {
    const double sv = -bq / (2.0 * a);
    if (sv > sa && sv < sb) {
      const double v = fma(sv, fma(sv, a, bq), c);
      lo = fmin(lo, v);
      hi = fmax(hi, v);
    }
  }
  const double ga = 1.0 / (2.0 * PI * du * fa), gb = 1.0 / (2.0 * PI * du * fb);
  tl = tc + fmin(lo * ga, lo * gb);
  th = tc + fmax(hi * ga, hi * gb);
}

// sin, cos of x, both reduction steps (|x| < 5e13), table entry from LDS
__device__ inline void sincos_tab(double x, double* s, double* c) {
  const double km = fma(x, kTabScale, kRoundMagic);
  const double k = km - kRoundMagic;
  sincos_tab_kr(km, fma(-k, kTabStepLo, fma(-k, kTabStepHi, x)), s, c);
}

// place of a tile's bin in the panel kernel's record (double2 [TILE / 32][PANEL_REC][32]: a half
// wave reads 512 consecutive bytes per entry, and a bin's entries lie within one load's offset)
__host__ __device__ inline int panel_rec_at(int q) { return (q >> 5) * (32 * PANEL_REC) + (q & 31); }

// BinPre of a panel's point from its stored values
__device__ inline void panel_point_pre(const DetectorDev& det, const double* __restrict__ pd, int k, int j, BinPre& b) {
  const double2* q = reinterpret_cast<const double2*>(pd + PAN_PT + k * PAN_PT_D);
  const double2 q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3], q4 = q[4];
  b.f = q0.x;
  b.j = j;
  b.pif = PI * b.f;
  b.xL = PI * b.f * det.L;
  b.hb1 = q0.y;
  b.hb2 = q1.x;
  b.hb3 = q1.y;
  b.he1 = q2.x;
  b.he2 = q2.y;
  b.he3 = q3.x;
  b.sxL = q3.y;
  b.cxL = q4.x;
}

// T components of one mode at one point (u = 1; without pf, pfT), and k.x0
template <int KIND>
__device__ inline void panel_point(const DetectorDev& det, const double* __restrict__ mf, const double* __restrict__ n0,
                                   const BinPre& b, const RowC& rc, double* one, double T[6], double& kx0) {
  ModeG g;
  mode_geom<0, KIND, 2>(det, mf, n0, b, rc, g, one);
  kx0 = g.kx0;
  Cx l[6];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    PairV v;
    pair_eval<0>(det, b, g, a, v);
    const int lp = a == 0 ? 2 : (a == 1 ? 4 : 0);
    l[lp] = scale(v.C, v.sp);
    l[lp + 1] = scale(v.C, v.sm);
  }
  const Cx D = {(b.cxL - b.sxL) * (b.cxL + b.sxL), -2.0 * b.sxL * b.cxL};  // exp(-2 i xL)
  const Cx X = add(sub(l[5], l[0]), mul(D, sub(l[4], l[1])));
  const Cx Y = add(sub(l[1], l[2]), mul(D, sub(l[0], l[3])));
  const Cx Z = add(sub(l[3], l[4]), mul(D, sub(l[2], l[5])));
  Cx o[3] = {X, Y, Z};
  if (det.orthogonal) {
    const double r2 = 0.70710678118654752440, r6 = 0.40824829046386301637;
    o[0] = scale(sub(Z, X), r2);
    o[1] = scale(add(sub(X, scale(Y, 2.0)), Z), r6);
    o[2] = add(add(sub(l[1], l[0]), sub(l[3], l[2])), sub(l[5], l[4]));
  }
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    T[2 * c] = o[c].re;
    T[2 * c + 1] = o[c].im;
  }
}

// adjoints of the six links from those of the channels (tile_rows, without pf and pfT)
__device__ inline void panel_link_adjoints(const DetectorDev& det, const BinPre& b, const Cx wch[3], Cx wl[6]) {
  Cx wX = wch[0], wY = wch[1], wZ = wch[2], wT = {0.0, 0.0};
  if (det.orthogonal) {
    const double r2 = 0.70710678118654752440, r6 = 0.40824829046386301637;
    wX = {fma(-r2, wch[0].re, r6 * wch[1].re), fma(-r2, wch[0].im, r6 * wch[1].im)};
    wY = scale(wch[1], -2.0 * r6);
    wZ = {fma(r2, wch[0].re, r6 * wch[1].re), fma(r2, wch[0].im, r6 * wch[1].im)};
    wT = wch[2];
  }
  const Cx cD = {(b.cxL - b.sxL) * (b.cxL + b.sxL), 2.0 * b.sxL * b.cxL};
  const Cx DWX = mul(cD, wX), DWY = mul(cD, wY), DWZ = mul(cD, wZ);
  wl[0] = sub(DWY, wX);
  wl[1] = sub(wY, DWX);
  wl[2] = sub(DWZ, wY);
  wl[3] = sub(wZ, DWY);
  wl[4] = sub(DWX, wZ);
  wl[5] = sub(wX, DWZ);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    wl[2 * a] = sub(wl[2 * a], wT);
    wl[2 * a + 1] = add(wl[2 * a + 1], wT);
  }
}

// LDS written by some lanes of a wave and read by others of the same wave: LDS operations of one
// wave execute in order, so only the compiler has to be kept from moving them
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

#define PANEL_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

// sum over the 32 lanes of each half wave
__device__ inline double half_sum(double v) {
  v = half_swap_sum<16>(v, v);
  v += dpp_mov<0x128>(v);
  v += dpp_mov<0x124>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0xB1>(v);
  return v;
}

// The unit phasors of a mode at a lane's bins, c2: its coefficients in LDS (entry 3 of row j: those
// of x^j in 2 pi k.x0 and of s^j in Psi).  All phases are reduced and their table entries requested
// before the first polynomial, so that the LDS latency is paid once
template <int NB>
__device__ __forceinline__ void panel_phasors(const double2* c2, const double* x, const double* s, double fmid,
                                              double fhalf, Cx* u) {
  double r[NB];
  double2 t[NB];
  {
    double2 cq[PANEL_K];
#pragma unroll
    for (int j = 0; j < PANEL_K; ++j) cq[j] = c2[4 * j + 3];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const double kx =
          fma(x[i], fma(x[i], fma(x[i], fma(x[i], cq[4].x, cq[3].x), cq[2].x), cq[1].x), cq[0].x);
      const double psi = fma(s[i], fma(s[i], fma(s[i], cq[3].y, cq[2].y), cq[1].y), cq[0].y);
      int k_lo;
      tab_reduce(fma(fma(x[i], fhalf, fmid), kx, psi), r[i], k_lo);
      t[i] = g_trig[k_lo & (kTrigN - 1)];
    }
  }
  PANEL_SCHED_FENCE();
#pragma unroll
  for (int i = 0; i < NB; ++i) {  // sincos_tab_kr's polynomials and rotation
    const double r2 = r[i] * r[i];
    const double sr = fma(r[i] * r2, fma(r2, 1.0 / 120.0, -1.0 / 6.0), r[i]);
    const double cr = fma(r2, fma(r2, fma(r2, -1.0 / 720.0, 1.0 / 24.0), -0.5), 1.0);
    u[i] = {fma(t[i].y, cr, -t[i].x * sr), -fma(t[i].x, cr, t[i].y * sr)};
  }
}

// places of a lane's bins in the panel (x) and in the node interval (s)
template <int NB>
__device__ __forceinline__ void panel_places(const double2* __restrict__ rec, int b0, int n, double fmid,
                                             double inv_half, int lane, double* s, double* x) {
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const double2 fs = rec[panel_rec_at(b0 + min((lane & 31) + 32 * i, n - 1))];
    s[i] = fs.y;
    x[i] = (fs.x - fmid) * inv_half;
  }
}

// Two rows (one per half wave; cf0: the first one's coefficients, h_stride (row, mode) pairs before
// the other's) of one panel, NB bins per lane: returns the lane's share of the row's lnL; GRAD:
// leaves the moments of every mode in the T slots.  alive: modes that reach the panel in either
// row (uniform)
template <bool GRAD, int NB>
__device__ __forceinline__ double panel_bins(int n_modes, unsigned alive, double* cf0, int h_stride, double* red, const double2* __restrict__ rec,
                                    int b0, int n, double fmid, double fhalf, double tc, const double* s,
                                    const double* x, int lane) {
  const int l32 = lane & 31;
  double* cf = cf0 + (lane >> 5) * h_stride * PANEL_CF;
  Cx acc[NB][3];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int c = 0; c < 3; ++c) acc[i][c] = {0.0, 0.0};
  // the scheduling fences keep the unrolled bins' temporaries apart: without them the scheduler
  // interleaves all eight and spills several hundred registers
  for (int m = 0; m < n_modes; ++m) {
    if (!((alive >> m) & 1u)) continue;
    const double2* c2 = reinterpret_cast<const double2*>(cf + m * PANEL_CF);
    Cx u[NB];
    panel_phasors<NB>(c2, x, s, fmid, fhalf, u);
    double2 tn[PANEL_K];  // the next channel's coefficients
#pragma unroll
    for (int j = 0; j < PANEL_K; ++j) tn[j] = c2[4 * j];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double2 t[PANEL_K];
#pragma unroll
      for (int j = 0; j < PANEL_K; ++j) t[j] = tn[j];
      if (c < 2) {
#pragma unroll
        for (int j = 0; j < PANEL_K; ++j) tn[j] = c2[4 * j + c + 1];
      }
      PANEL_SCHED_FENCE();
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        double tr = t[PANEL_K - 1].x, ti = t[PANEL_K - 1].y;
#pragma unroll
        for (int j = PANEL_K - 2; j >= 0; --j) {
          tr = fma(tr, x[i], t[j].x);
          ti = fma(ti, x[i], t[j].y);
        }
        acc[i][c].re = fma(u[i].re, tr, fma(-u[i].im, ti, acc[i][c].re));
        acc[i][c].im = fma(u[i].re, ti, fma(u[i].im, tr, acc[i][c].im));
      }
      PANEL_SCHED_FENCE();
    }
  }
  double v = 0.0;
  double2 nx[PANEL_REC];  // the next bin's record, requested while this one is worked on
  auto load_rec = [&](int i) {
    const double2* rq = rec + panel_rec_at(b0 + min(l32 + 32 * i, n - 1));
#pragma unroll
    for (int k = 0; k < PANEL_REC; ++k) nx[k] = rq[32 * k];
  };
  load_rec(0);
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    double2 r[PANEL_REC];
#pragma unroll
    for (int k = 0; k < PANEL_REC; ++k) r[k] = nx[k];
    if (i + 1 < NB) load_rec(i + 1);
    PANEL_SCHED_FENCE();
    const bool in = l32 + 32 * i < n;
    const double w[3] = {in ? r[1].x : 0.0, in ? r[2].y : 0.0, in ? r[4].x : 0.0};
    const Cx d[3] = {{r[1].y, r[2].x}, {r[3].x, r[3].y}, {r[4].y, r[5].x}};
    double se, ce;
    sincos_tab(2.0 * (PI * r[0].x) * tc, &se, &ce);  // 2 pi f t_c rounded once, as the reference's own factor
    const Cx e = {ce, -se};
    const Cx P = mul(Cx{r[5].y, r[6].x}, e), PT = mul(Cx{r[6].y, r[7].x}, e);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const Cx Pc = c == 2 ? PT : P;
      const Cx o = mul(Pc, acc[i][c]);
      const Cx q = {d[c].re - o.re, d[c].im - o.im};
      v -= w[c] * fma(q.re, q.re, q.im * q.im);
      if constexpr (GRAD) {
        acc[i][c] = mul(Cx{2.0 * w[c] * q.re, -2.0 * w[c] * q.im}, Pc);
        asm volatile("" : "+v"(acc[i][c].re), "+v"(acc[i][c].im) : : "memory");  // formed here, not at its use
      }
    }
    asm volatile("" : "+v"(v) : : "memory");
    PANEL_SCHED_FENCE();
  }
  if constexpr (GRAD) {
    for (int m = 0; m < n_modes; ++m) {
      if (!((alive >> m) & 1u)) continue;
      double* cm = cf + m * PANEL_CF;
      const double2* c2 = reinterpret_cast<const double2*>(cm);
      Cx u[NB];
      panel_phasors<NB>(c2, x, s, fmid, fhalf, u);
      PANEL_SCHED_FENCE();
      // moments of one channel at a time (20 registers of sums instead of 60), [j][re, im]
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        double M[2 * PANEL_K];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
          const Cx g = mul(acc[i][c], u[i]);
          const double x2 = x[i] * x[i];
          const double xp[PANEL_K] = {1.0, x[i], x2, x2 * x[i], x2 * x2};
          if (i == 0) {
            M[0] = g.re;
            M[1] = g.im;
#pragma unroll
            for (int j = 1; j < PANEL_K; ++j) {
              M[2 * j] = g.re * xp[j];
              M[2 * j + 1] = g.im * xp[j];
            }
          } else {
            M[0] += g.re;
            M[1] += g.im;
#pragma unroll
            for (int j = 1; j < PANEL_K; ++j) {
              M[2 * j] = fma(g.re, xp[j], M[2 * j]);
              M[2 * j + 1] = fma(g.im, xp[j], M[2 * j + 1]);
            }
          }
          if (i & 1) PANEL_SCHED_FENCE();
        }
        // rows of 16 lanes trade halves of the ten sums
#pragma unroll
        for (int k = 0; k < PANEL_K; ++k)
          red[(PANEL_K * c + k) * PANEL_RED + lane] = half_swap_sum<16>(M[k], M[PANEL_K + k]);
        PANEL_SCHED_FENCE();
      }
      wave_sync();
      // lane t < 60: the 16 lanes of sum t mod 30 of row t / 30, stored over the row's T slots
      if (lane < 60) {
        const int hh = lane >= 30 ? 1 : 0, k = lane - 30 * hh, c = k / 10, kk = k - 10 * c, q = kk >= 5 ? 1 : 0;
        const double2* p =
            reinterpret_cast<const double2*>(red + (PANEL_K * c + kk - 5 * q) * PANEL_RED + 32 * hh + 16 * q);
        double2 z[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) z[j] = p[j];
#pragma unroll
        for (int j = 4; j; j >>= 1)
#pragma unroll
          for (int i = 0; i < j; ++i) {
            z[i].x += z[i + j].x;
            z[i].y += z[i + j].y;
          }
        // kk = 2 j + (re, im): component 2 c + (re, im) of x^j
        cf0[(hh * h_stride + m) * PANEL_CF + 8 * (kk >> 1) + 2 * c + (kk & 1)] = z[0].x + z[0].y;
      }
      wave_sync();
    }
  }
  return v;
}

// Persistent kernel over a tile range.  Every wave takes work items of its own (group of tiles x
// PANEL_ROWS rows; small batches, grp null: one panel x PANEL_ROWS rows) and needs no other wave: rows are summed over the item's tiles in order, so a
// row's result does not depend on its batch.  Stores the item's partial sums (zero for the tiles
// and rows that go bin by bin, which k_lnl adds).  KIND: the orbit kind (a duty-cycled detector's
// panels lie on its window's plateau).  dbits [P][words]: bit 1 the (tile, row) goes bin by bin;
// off_bits: the tile's response is zero
template <bool GRAD, int KIND>
__global__ __launch_bounds__(TILE, 2) void k_lnl_panel(
    const DetectorDev* __restrict__ dets, int n_det, int n_tiles, const double* __restrict__ tile_f0,
    const double* __restrict__ tile_dd, const int* __restrict__ grp, int n_grp, const double* __restrict__ pconst,
    const double* __restrict__ nodes, const double* __restrict__ nodes_grad, int NNS, double du, ModeList modes, int P,
    int group_offset, int* __restrict__ work_counter,
    double* __restrict__ partial, const unsigned long long* __restrict__ off_bits,
    const unsigned long long* __restrict__ dbits, PanelDev pan, int pan_begin) {
  constexpr int NOUT = GRAD ? 1 + PES_N_PARAMS : 1;
  constexpr int NW = TILE / 64;
  __shared__ double acc_all[NW][2][PANEL_ROWS * NOUT];  // per wave: the item's sums, the tile's
  __shared__ __align__(16) double cf_all[NW][PANEL_PAIRS * PANEL_CF];
  __shared__ __align__(16) double red_all[GRAD ? NW : 1][GRAD ? 16 * PANEL_RED : 1];
  __shared__ __align__(16) double one[2];
  __shared__ double ci[PANEL_K][PANEL_K];
  if (threadIdx.x < 2) one[threadIdx.x] = threadIdx.x == 0 ? 1.0 : 0.0;
  if (threadIdx.x < PANEL_K * PANEL_K) {
    const int j = threadIdx.x / PANEL_K, k = threadIdx.x % PANEL_K;
    ci[j][k] = panel_ci(j, k);
  }
  trig_table_load();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nm = modes.n;
  const int nrh = panel_rows_half(nm), nr = 2 * nrh;
  double* cf = cf_all[wave];
  double* red = red_all[GRAD ? wave : 0];
  const int words = (n_tiles + 63) >> 6;
  double* acc = acc_all[wave][0];
  double* tacc = acc_all[wave][1];
  const int n_chunks = (P + PANEL_ROWS - 1) / PANEL_ROWS;
  const int n_work = n_chunks * n_grp;
  // items from a queue; those of small batches, a panel each, dealt out beforehand (a queue hands out
  // one per ~11 ns: 90 us for a year of LISA data)
  int next = blockIdx.x * NW + wave;
  for (;;) {
    int w = next;
    if (grp) {
      if (lane == 0) w = atomicAdd(work_counter, 1);
      w = __builtin_amdgcn_readfirstlane(w);
    }
    next += gridDim.x * NW;
    if (w >= n_work) break;
    const int gl = w / n_chunks, c = w % n_chunks;
    const int p0 = c * PANEL_ROWS, p1 = min(P, p0 + PANEL_ROWS);
    for (int i = lane; i < 2 * PANEL_ROWS * NOUT; i += 64) acc[i] = 0.0;
    wave_sync();
    const int one_pan = pan_begin + gl;  // grp null: the item is one panel
    const int t_first = grp ? grp[gl] : pan.pan_i[4 * one_pan + 3], t_end = grp ? grp[gl + 1] : t_first + 1;
    for (int tile = t_first; tile < t_end; ++tile) {
      const int pan0 = pan.tile_pan[2 * tile], np = pan.tile_pan[2 * tile + 1];
      if (np == 0) continue;
      const int pan_a = grp ? pan0 : one_pan, pan_b = grp ? pan0 + np : one_pan + 1;
      const double f0 = tile_f0[tile];
      // lane <-> row of the item: evaluated, zero over the whole tile, or left to the other kernel
      bool act = false;
      if (p0 + lane < p1) {
        const int p = p0 + lane;
        const double* pc = pconst + (size_t)p * PC_STRIDE;
        const size_t wd = (size_t)p * words + (tile >> 6);
        const unsigned long long db = dbits[wd], ob = off_bits ? off_bits[wd] : 0ull;
        const bool zero = f0 > pc[PC_FCUT] || ((ob >> (tile & 63)) & 1ull) != 0;
        if (pc[PC_VALID] != 0.0) {
          if (zero && pan_a == pan0) acc[lane * NOUT] -= tile_dd[tile];
          act = !zero && ((db >> (tile & 63)) & 1ull) == 0;
        }
      }
      const unsigned act_rows = (unsigned)__ballot(act);
      if (act_rows == 0u) continue;
      for (int r0 = p0; r0 < p1; r0 += nr) {
      const unsigned active = (act_rows >> (r0 - p0)) & ((1u << nr) - 1u);
      if (active == 0u) continue;
      const DetectorDev& det = dets[tile_detector(dets, n_det, tile)];
      const double2* rec_t = pan.rec + (size_t)tile * PANEL_REC * TILE;
      for (int pi = pan_a; pi < pan_b; ++pi) {
        const double* pd = pan.pan_d + (size_t)pi * PAN_D;
        const int j0 = pan.pan_i[4 * pi], b0 = pan.pan_i[4 * pi + 1], n = pan.pan_i[4 * pi + 2];
        // geometry lanes: (row of the half, mode, point); lanes past the last repeat it and store
        // nothing.  Formed anew per use (gl_of): held over the bins' loops they were spilled
        struct GeoLane {
          int row, m, k;
          bool on;
        };
        auto gl_of = [&]() -> GeoLane {
          int ln = lane;
          asm volatile("" : "+v"(ln));
          const int l32 = ln & 31, seg = min(l32 / (PANEL_K * nm), nrh - 1);
          const int rem = min(l32 - seg * PANEL_K * nm, PANEL_K * nm - 1);
          const int m = rem / PANEL_K;
          return {(ln >> 5) * nrh + seg, m, rem - PANEL_K * m, l32 < nrh * PANEL_K * nm};
        };
        unsigned long long alive_l;
        {  // coefficients of every (row, mode)
          const GeoLane g = gl_of();
          const int my_row = min(r0 + g.row, p1 - 1);
          const double* pcg = pconst + (size_t)my_row * PC_STRIDE;
          const double* mf = pcg + PC_MODE + g.m * PC_MODE_STRIDE;
          const double* n0 = nodes + (((size_t)my_row * nm + g.m) * NNS + j0) * 4;
          double* cfl = cf + (g.row * nm + g.m) * PANEL_CF;
          const bool alive_me = !(f0 > mf[MF_CUT]);
          alive_l = __ballot(alive_me);
          BinPre b;
          panel_point_pre(det, pd, g.k, j0, b);
          RowC rc = load_row(pcg, b);
          if constexpr (kGeo<KIND>) row_geo(det, rc);
          double T[6], kx0;
          panel_point<KIND>(det, mf, n0, b, rc, one, T, kx0);
          if (g.on) {
#pragma unroll
            for (int i = 0; i < 6; ++i) cfl[8 * g.k + i] = alive_me ? T[i] : 0.0;
            cfl[8 * g.k + 6] = 2.0 * PI * kx0;
          }
          wave_sync();
          double cs[7];
#pragma unroll
          for (int i = 0; i < 7; ++i) cs[i] = 0.0;
#pragma unroll
          for (int k = 0; k < PANEL_K; ++k) {
            const double a = ci[g.k][k];
#pragma unroll
            for (int i = 0; i < 7; ++i) cs[i] = fma(a, cfl[8 * k + i], cs[i]);
          }
          // Psi as a cubic in s
          const double dP = n0[6] - n0[2], m0 = du * n0[3], m1 = du * n0[7];
          const double ps = g.k == 0 ? n0[2]
                                     : (g.k == 1 ? m0 : (g.k == 2 ? 3.0 * dP - 2.0 * m0 - m1
                                                                  : (g.k == 3 ? m0 + m1 - 2.0 * dP : 0.0)));
          wave_sync();
          if (g.on) {
#pragma unroll
            for (int i = 0; i < 7; ++i) cfl[8 * g.k + i] = cs[i];
            cfl[8 * g.k + 7] = ps;
          }
          wave_sync();
        }
        // the rows two by two, the bins' places once for all of them
        auto row_pairs = [&](auto nbc) {
          constexpr int NB = decltype(nbc)::value;
          for (int rp = 0; rp < nrh; ++rp) {
            const bool on_a = (active >> rp) & 1u, on_b = (active >> (nrh + rp)) & 1u;
            if (!on_a && !on_b) continue;
            unsigned alive = 0;  // modes that reach the tile in either row
            for (int m = 0; m < nm; ++m) {
              const int bit = (rp * nm + m) * PANEL_K;
              alive |= (unsigned)(((alive_l >> bit) | (alive_l >> (32 + bit))) & 1ull) << m;
            }
            double s[NB], x[NB];
            // addresses are formed per pair of rows: hoisted out of the loops they were spilled
            int ln = lane;
            asm volatile("" : "+v"(ln));
            panel_places<NB>(rec_t, b0, n, pd[0], pd[1], ln, s, x);
            const int h = ln >> 5;
            const double tc = pconst[(size_t)min(r0 + h * nrh + rp, p1 - 1) * PC_STRIDE + PC_TC];
            double v = panel_bins<GRAD, NB>(nm, alive, cf + rp * nm * PANEL_CF, nrh * nm, red, rec_t, b0, n, pd[0], pd[2],
                                            tc, s, x, ln);
            v = half_sum(v);
            if ((ln & 31) == 0 && (h ? on_b : on_a)) tacc[(r0 + h * nrh + rp - p0) * NOUT] += v;
          }
        };
        if (n > 128)
          row_pairs(std::integral_constant<int, 8>());
        else if (n > 64)
          row_pairs(std::integral_constant<int, 4>());
        else
          row_pairs(std::integral_constant<int, 2>());
        if constexpr (GRAD) {
          const GeoLane g = gl_of();
          const int my_row = min(r0 + g.row, p1 - 1);
          const double* pcg = pconst + (size_t)my_row * PC_STRIDE;
          const double* mf = pcg + PC_MODE + g.m * PC_MODE_STRIDE;
          const size_t nrow = ((size_t)my_row * nm + g.m) * NNS + j0;
          const double* cfl = cf + (g.row * nm + g.m) * PANEL_CF;
          Cx wch[3];
#pragma unroll
          for (int cc = 0; cc < 3; ++cc) wch[cc] = {0.0, 0.0};
#pragma unroll
          for (int j = 0; j < PANEL_K; ++j) {  // ell_k(x) = sum_j ci[j][k] x^j
            const double a = ci[j][g.k];
#pragma unroll
            for (int cc = 0; cc < 3; ++cc) {
              wch[cc].re = fma(a, cfl[8 * j + 2 * cc], wch[cc].re);
              wch[cc].im = fma(-a, cfl[8 * j + 2 * cc + 1], wch[cc].im);
            }
          }
          BinPre b;
          panel_point_pre(det, pd, g.k, j0, b);
          RowC rc = load_row(pcg, b);
          if constexpr (kGeo<KIND>) row_geo(det, rc);
          Cx wl[6];
          panel_link_adjoints(det, b, wch, wl);
          AdjAcc aa;
          aa.pb = aa.qb = aa.kb = V3{0.0, 0.0, 0.0};
#pragma unroll
          for (int i = 0; i < 4; ++i) aa.gint[i] = 0.0;
          aa.gh_re = aa.mphi = aa.iota = aa.tc = 0.0;
          mode_adjoint<0, KIND>(det, mf, modes.id[g.m], nodes + nrow * 4, nodes_grad + nrow * 16, b, rc, wl, pcg, aa,
                                one);
          double G[PES_N_PARAMS];
#pragma unroll
          for (int i = 0; i < 4; ++i) G[i] = aa.gint[i];
          G[4] = -aa.gh_re * pcg[PC_INVDL];
          G[5] = -aa.mphi;
          G[6] = aa.iota;
          const V3 dlp = {pcg[PC_DLP], pcg[PC_DLP + 1], pcg[PC_DLP + 2]};
          const V3 dlq = {pcg[PC_DLQ], pcg[PC_DLQ + 1], pcg[PC_DLQ + 2]};
          const V3 dlk = {pcg[PC_DLK], pcg[PC_DLK + 1], pcg[PC_DLK + 2]};
          G[7] = dot3(aa.pb, dlp) + dot3(aa.qb, dlq) + dot3(aa.kb, dlk);
          const V3 dbp = {pcg[PC_DBP], pcg[PC_DBP + 1], pcg[PC_DBP + 2]};
          const V3 dbq = {pcg[PC_DBQ], pcg[PC_DBQ + 1], pcg[PC_DBQ + 2]};
          const V3 dbk = {pcg[PC_DBK], pcg[PC_DBK + 1], pcg[PC_DBK + 2]};
          G[8] = dot3(aa.pb, dbp) + dot3(aa.qb, dbq) + dot3(aa.kb, dbk);
          G[9] = dot3(aa.pb, rc.q) - dot3(aa.qb, rc.p);
          G[10] = aa.tc;
          const bool alive_me = !(f0 > mf[MF_CUT]);
          wave_sync();
#pragma unroll
          for (int i = 0; i < PES_N_PARAMS; ++i) red[lane * PANEL_G + i] = alive_me ? G[i] : 0.0;
          wave_sync();
          // lane <-> (row, parameter): the sum over the row's modes and points
          for (int idx = lane; idx < nr * PES_N_PARAMS; idx += 64) {
            const int rg = idx / PES_N_PARAMS, o = idx - rg * PES_N_PARAMS;
            if ((active >> rg) & 1u) {
              const int hh = rg >= nrh ? 1 : 0;
              const double* p = red + (32 * hh + (rg - hh * nrh) * PANEL_K * nm) * PANEL_G + o;
              double sum = 0.0;
              for (int m = 0; m < nm; ++m, p += PANEL_K * PANEL_G)
                sum += ((p[0] + p[PANEL_G]) + (p[2 * PANEL_G] + p[3 * PANEL_G])) + p[4 * PANEL_G];
              tacc[(r0 + rg - p0) * NOUT + 1 + o] += sum;
            }
          }
          wave_sync();
        }
      }
      }
      wave_sync();
      // the tile's sums onto the item's, tile by tile
      for (int i = lane; i < PANEL_ROWS * NOUT; i += 64) {
        acc[i] += tacc[i];
        tacc[i] = 0.0;
      }
      wave_sync();
    }
    for (int i = lane; i < (p1 - p0) * NOUT; i += 64) {
      const int pl = i / NOUT, o = i - pl * NOUT;
      partial[((size_t)(group_offset + gl) * NOUT + o) * P + p0 + pl] = acc[i];
    }
    wave_sync();
  }
}

// The panel kernel's record of every bin: (f, s), (w0, Re d0), (Im d0, w1), d1, (w2, Re d2), (Im d2, Re p0), (Im p0, Re p2),
// (Im p2, 0), with the channels' prefactors p0 = p1 and p2 (pfT for A/E/T).  One launch per detector.
__global__ __launch_bounds__(TILE) void k_panel_rec(const DetectorDev* __restrict__ dets, int det_i,
                                                    const double* __restrict__ bin_f, const double* __restrict__ bin_s,
                                                    const int* __restrict__ bin_j, const double* __restrict__ bin_rec,
                                                    double du, double2* __restrict__ rec) {
  const DetectorDev& det = dets[det_i];
  const int bi = det.bin_offset + blockIdx.x * TILE + threadIdx.x;
  BinPre b;
  bin_prepare(det, bin_f[bi], bin_s[bi], bin_j[bi], du, b);
  TdiC t;
  tdi_consts(det, b, t);
  const double* r = bin_rec + (size_t)bi * BIN_REC;
  const Cx p2 = det.orthogonal ? t.pfT : t.pf;
  double2* o = rec + (size_t)(bi / TILE) * PANEL_REC * TILE + panel_rec_at(threadIdx.x);
  o[0] = make_double2(bin_f[bi], bin_s[bi]);
  o[32] = make_double2(r[0], r[1]);
  o[64] = make_double2(r[2], r[3]);
  o[96] = make_double2(r[4], r[5]);
  o[128] = make_double2(r[6], r[7]);
  o[160] = make_double2(r[8], t.pf.re);
  o[192] = make_double2(t.pf.im, p2.re);
  o[224] = make_double2(p2.im, 0.0);
}

// Per (tile, row): bit 1 when the pair goes bin by bin: the tile has no panels, a mode's cut lies
// inside it, a mode's orbit angle (geocentric: the rotation angle) turns by more than PANEL_SWING
// over a panel, or a duty-cycled detector's window is not flat 1 over a panel (off tiles aside:
// their response is zero).  One wave per 64 tiles writes the row's word with a vote; the tiles and
// groups with any such row are marked, and the groups listed, for the bin-by-bin kernel (in an order
// that depends on the scheduling; every group's sums are its own).
__global__ __launch_bounds__(64) void k_panel_class(const DetectorDev* __restrict__ dets, int n_det, int n_tiles,
                                                    const double* __restrict__ tile_f0, const double* __restrict__ bin_f,
                                                    const double* __restrict__ pconst, const double* __restrict__ nodes,
                                                    int NNS, double du, ModeList modes, int P, int words,
                                                    const unsigned long long* __restrict__ off_bits, PanelDev pan,
                                                    BinWork bw, TileGroups rb, int fine,
                                                    unsigned long long* __restrict__ dbits) {
  const int tile = blockIdx.x * 64 + threadIdx.x;
  const int tl_ = min(tile, n_tiles - 1);
  const int np = tile < n_tiles ? pan.tile_pan[2 * tile + 1] : 0, pp0 = pan.tile_pan[2 * tl_];
  const double f0 = tile_f0[tl_], f1 = bin_f[(size_t)tl_ * TILE + TILE - 1];
  const DetectorDev& det = dets[tile_detector(dets, n_det, tl_)];
  const int epoch = bw.state[0];
  const double wmax = det.kind == 1 ? fmax(fabs(det.omega_rot), kOmegaYear) : kOmegaYear;
  for (int p = blockIdx.y; p < P; p += gridDim.y) {
    const double* pc = pconst + (size_t)p * PC_STRIDE;
    bool direct = np == 0 && tile < n_tiles;
    const bool zero = f0 > pc[PC_FCUT] || pc[PC_VALID] == 0.0 ||
                      (off_bits && ((off_bits[(size_t)p * words + blockIdx.x] >> threadIdx.x) & 1ull) != 0);
    if (np > 0 && !zero) {
      const double tc = pc[PC_TC];
      for (int mi = 0; mi < modes.n && !direct; ++mi) {
        const double cut = pc[PC_MODE + mi * PC_MODE_STRIDE + MF_CUT];
        if (f0 > cut) continue;
        if (f1 > cut) direct = true;
        const double* nm = nodes + ((size_t)p * modes.n + mi) * NNS * 4;
        for (int k = pp0; k < pp0 + np && !direct; ++k) {
          const double* pd = pan.pan_d + (size_t)k * PAN_D;
          double tl, th;
          panel_t_range(nm + (size_t)pan.pan_i[4 * k] * 4, pd[0] - pd[2], pd[0] + pd[2], pd[3], pd[4], du, tc, tl, th);
          if (!((th - tl) * wmax <= PANEL_SWING)) direct = true;  // NaN goes bin by bin
          if (det.duty) {
            const double m = 1e-3 + 1e-9 * (fabs(tl) + fabs(th));
            const double start =
                det.duty_t0 + floor((tl - m - det.duty_t0) * det.duty_inv_period) * det.duty_period;
            if (!(tl - m - start >= det.duty_taper && th + m - start <= det.duty_on - det.duty_taper)) direct = true;
          }
        }
      }
    }
    const unsigned long long word = __ballot(direct);
    if (threadIdx.x == 0) dbits[(size_t)p * words + blockIdx.x] = word;
    if (direct && bw.tile_any[tile] != epoch) {
      bw.tile_any[tile] = epoch;
      const int r = bw.tile_range[tile], base = fine ? rb.tile0[r] : rb.group0[r];
      const int g = fine ? tile : bw.tile_group[tile];
      if (atomicExch(bw.group_any + g, epoch) != epoch) bw.list[base + atomicAdd(bw.state + 1 + r, 1)] = g - base;
    }
  }
}
