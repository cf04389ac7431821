// The order in which the blocks of a product take its tiles (gemm_bf16.hip, gemm_f32.hip).
#pragma once
#include "common.h"

// Which tile a block works on.  Blocks go to the eight dies (each with an L2 of
// its own) in turn, so block b runs on die b % 8.  The tiles are put in an
// order in which neighbours share operands (panels of PANEL rows of tiles; in
// a panel column after column) and that sequence is cut into eight runs of
// equal length, one a die.  So every die gets the same number of tiles to
// within one (dealing whole groups of tiles left a die with 40 tiles and
// another with 4 at 2,056 rows), and the blocks at work on a die at one time
// are a few columns of one panel: what one brings into the L2 the others find
// there.  Returns false for the padding blocks of the grid.
template <int PANEL>
__device__ __forceinline__ bool tile_of_block(int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n, run = (total + 7) / 8;
  const int die = blockIdx.x & 7, local = blockIdx.x >> 3;
  const int idx = die * run + local;
  if (local >= run || idx >= total) return false;
  const int panel = min(idx / (PANEL * tiles_n), (tiles_m + PANEL - 1) / PANEL - 1);  // (only the last is short)
  const int rem = idx - panel * PANEL * tiles_n;
  const int h = min(PANEL, tiles_m - panel * PANEL);
  tn = rem / h;
  tm = panel * PANEL + rem % h;
  return true;
}

// The columns of tiles that a die's run touches, panel after panel: `n` of them from column `first` of the sequence in which panel
// after panel brings its columns (the matrix's column is the remainder by tiles_n).
template <int PANEL>
__device__ __forceinline__ bool columns_of_die(int tiles_m, int tiles_n, int die, int& first, int& n) {
  const int total = tiles_m * tiles_n, run = (total + 7) / 8;
  if (die * run >= total) return false;
  const auto column_of = [&](int idx) {
    const int panel = min(idx / (PANEL * tiles_n), (tiles_m + PANEL - 1) / PANEL - 1);
    return panel * tiles_n + (idx - panel * PANEL * tiles_n) / min(PANEL, tiles_m - panel * PANEL);
  };
  first = column_of(die * run);
  n = column_of(min(total, (die + 1) * run) - 1) - first + 1;
  return true;
}
