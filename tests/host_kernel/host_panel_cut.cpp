// panel_cut on the grids of tests/test_host_panel_cut.py.  Input file: int32 n, n frequencies and n
// int32 node intervals, the arm length in seconds.  Prints, per tile of 256 bins, the number of
// panels and (first bin, bins, node interval) of each.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "panel_cut.hpp"

int main(int argc, char** argv) {
  std::FILE* fh = argc > 1 ? std::fopen(argv[1], "rb") : nullptr;
  std::int32_t n = 0;
  if (!fh || std::fread(&n, 4, 1, fh) != 1 || n < 1) return 2;
  std::vector<double> f(n);
  std::vector<int> j(n);
  double L = 0.0;
  if (std::fread(f.data(), 8, n, fh) != (size_t)n || std::fread(j.data(), 4, n, fh) != (size_t)n ||
      std::fread(&L, 8, 1, fh) != 1)
    return 2;
  std::fclose(fh);
  for (int t = 0; t < n; t += 256) {
    pes::PanelCut p[pes::PANEL_MAX_PIECES];
    const int np = pes::panel_cut(&f[t], &j[t], n - t < 256 ? n - t : 256, L, p);
    std::printf("%d", np);
    for (int k = 0; k < np; ++k) std::printf(" %d %d %d", p[k].first, p[k].bins, p[k].node);
    std::printf("\n");
  }
  return 0;
}
