// Definitions shared by the kernels of pespace_amd.hip and hotpath.hpp: tile and chunk sizes,
// the per-row constant block, and the tile -> detector map.  Included inside the anonymous
// namespace of pespace_amd.hip.
#pragma once

constexpr int TILE = 256;      // bins per tile = threads per block
// parameter rows per work item of the gradient kernel (48: the most that leaves two blocks per
// CU the LDS for the staged node rows, the accumulators and the forward pass's unit phasors)
// and of the lnL-only one (160: 1.1% faster than 256)
template <bool GRAD>
constexpr int chunk_rows() { return GRAD ? 48 : 160; }
// default schedule: tiles per work item (8: the fastest in every timed schedule table of the
// one-year network, 4-7% ahead of 32 on 512-row samples) ...
constexpr int TILES_PER_GROUP = 8;
constexpr int MAX_TILES_PER_GROUP = 4096;
constexpr int BLOCKS_PER_CU = 4;     // ... and persistent blocks launched per CU
constexpr int MAX_MODES = 6;         // modes per context (ModeList)
// node rows per tile that the fused kernel stages in LDS (tiles spanning more read them from
// global memory): a 256-bin tile of a one-year grid spans at most 1.3e-3 Hz / f + 1 of the 1024
// log-spaced node intervals over 1e-4 - 0.06 Hz, under 16 above 1e-4 Hz
constexpr int NJ_STAGE = 16;
constexpr int BIN_REC = 10;          // doubles per bin of the fused kernel's weight and data record
constexpr int MAX_TILE_RANGES = 16;  // runs of detectors by duty flag per context
// fused-kernel launches per batch: one per range, and a second for a duty-cycled range (its work
// items on the window's plateau run in the plain instantiation), each with its own work counter;
// a third set flags the duty-cycled ranges with items that need the window (k_duty_items)
// and a fourth serves the panel kernel's launches
constexpr int N_WORK_COUNTERS = 4 * MAX_TILE_RANGES;

// ---- per-row constant block ------------------------------------------------------------
enum PConst {
  PC_TC = 0, PC_INVDL, PC_VALID, PC_DL,
  PC_P = 4, PC_Q = 7, PC_K = 10,
  PC_DLP = 13, PC_DLQ = 16, PC_DBP = 19, PC_DBQ = 22, PC_DLK = 25, PC_DBK = 28,
  PC_MODE = 32,  // per mode: Fp re,im, 2 Fc re,im, cut_hz, dFp/diota re,im, 2 dFc/diota re,im
  PC_MODE_STRIDE = 9,
  PC_FCUT = 32 + 6 * 9,  // largest mode cut [Hz]: the response is zero above it
  PC_OFFANY,             // 1: a tile of a duty-cycled detector lies in an off period for this row
  PC_STRIDE = 32 + 6 * 9 + 2
};
enum { MF_FPR = 0, MF_FPI, MF_FCR, MF_FCI, MF_CUT, MF_DFPR, MF_DFPI, MF_DFCR, MF_DFCI };

// ---- tile groups -----------------------------------------------------------------------
// The groups (RangeGroups) of all tile ranges in turn (range r: tiles tile0[r] .., groups group0[r] ..)
struct TileGroups {
  const int* first;
  int per, n_ranges, tile0[MAX_TILE_RANGES + 1], group0[MAX_TILE_RANGES];
  __device__ void tiles(int g, int& t0, int& t1) const {
    if (first) {
      t0 = first[g];
      t1 = first[g + 1];
      return;
    }
    int r = 0;
    while (r + 1 < n_ranges && group0[r + 1] <= g) ++r;
    t0 = tile0[r] + (g - group0[r]) * per;
    t1 = min(tile0[r + 1], t0 + per);
  }
};

// Rows per work item of the bin-by-bin kernel where panels leave it a list of n_list groups: the host's
// `rows`, chosen for the tiles without panels, and more where a small batch sends more its way (light
// systems, whose orbit turns too fast for panels), so that about `want` items remain (0: the host's).  A year
// of LISA data, 8 rows of 30 solar masses with the gradient: 0.95 -> 0.68 ms; all tiles bin by bin 0.86.
// At most 24, 48 with one or two modes: the last items end together, and an item's rows share the tile's
// preparation (lnL, ms, with 160, 48 and 24: LISA, 5e6 s, six modes, 300 rows from the prior 2.99, 2.63, 2.32;
// TianQin, 6e6 s, duty-cycled, 22 mode, 400 rows 0.97, 0.86, 1.03; with the gradient 24 for 48 rows: 6.26 ->
// 5.75 and 1.52 -> 1.64)
__device__ inline int listed_rows(int rows, int P, int n_list, int want, int n_modes) {
  return want > 0 ? max(rows, min(n_modes < 3 ? 48 : 24, (int)((long long)P * n_list / want))) : rows;
}

// detector owning tile `tile` (detectors are concatenated in tile order)
__device__ inline int tile_detector(const DetectorDev* dets, int n_det, int tile) {
  int acc = 0;
  for (int d = 0; d < n_det; ++d) {
    acc += dets[d].n_tiles;
    if (tile < acc) return d;
  }
  return n_det - 1;
}
