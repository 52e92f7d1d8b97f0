// Where a tile's bins are cut into panels (panel.hpp).  Host code.
#pragma once

#include <algorithm>
#include <cmath>

namespace pes {

constexpr double PANEL_EPS = 1.4e-3;    // relative half-width of a panel, at most
constexpr double PANEL_SWING = 3.0e-3;  // 2 pi (2 L) (f_hi - f_lo) and the orbit angles' turn, at most
// tiles cut into more panels go bin by bin: a panel costs its points whatever its bins (a year of
// the network, 1024 rows with the gradient: 5 panels at most 109.6 ms, 8 109.3, 12 110.3)
constexpr int PANEL_MAX_PIECES = 8;

struct PanelCut {
  int first, bins, node;  // first bin in the tile, number of bins, node interval
};

// How many widths at the bounds the frequencies lo .. hi take; L: arm length in seconds
inline double panel_widths(double lo, double hi, double L) {
  return std::max((hi - lo) / ((hi + lo) * PANEL_EPS), 4.0 * 3.14159265358979323846 * L * (hi - lo) / PANEL_SWING);
}

// The panels of a tile's nb bins (frequencies f increasing, node intervals j): cut at every node
// interval's end, and each part into as few panels of equal numbers of bins as its width needs.
// Where the bins are spaced unevenly (a gap, a change of spacing) and one of those is wider than the
// bounds, the part is cut by frequency instead, each panel as wide as the bounds allow.  Returns
// their number, 0 when it would be more than PANEL_MAX_PIECES.
inline int panel_cut(const double* f, const int* j, int nb, double L, PanelCut out[PANEL_MAX_PIECES]) {
  int np = 0;
  for (int a = 0, e; a < nb; a = e) {
    for (e = a + 1; e < nb && j[e] == j[a];) ++e;
    const double w = panel_widths(f[a], f[e - 1], L);
    const int k = w < (double)(e - a) ? std::max(1, (int)std::ceil(w)) : e - a;
    auto edge = [&](int i) { return a + (int)((long long)(e - a) * i / k); };
    bool even = np + k <= PANEL_MAX_PIECES;
    for (int i = 0; i < k && even; ++i) even = panel_widths(f[edge(i)], f[edge(i + 1) - 1], L) <= 1.0;
    if (even) {
      for (int i = 0; i < k; ++i) out[np++] = {edge(i), edge(i + 1) - edge(i), j[a]};
      continue;
    }
    for (int b = a, n; b < e; b += n) {
      for (n = 1; b + n < e && panel_widths(f[b], f[b + n], L) <= 1.0;) ++n;
      if (np == PANEL_MAX_PIECES) return 0;
      out[np++] = {b, n, j[a]};
    }
  }
  return np;
}

}  // namespace pes
