// How the rows of an expert's slice are cut into tiles; plain C++, so that host code can include it.
#pragma once
#ifdef __HIPCC__
#define EIA_MOE_HD __host__ __device__ __forceinline__
#else
#define EIA_MOE_HD inline
#endif

struct MoeTile {
  int lo, mu;                              // 64-row units lo .. lo + mu - 1 of the slice
};

// M tiles of a slice: as few as tiles of up to max_mu units allow.
EIA_MOE_HD int moe_slice_tiles(int rows, int max_mu) { return (rows + 64 * max_mu - 1) / (64 * max_mu); }

// Tile t of them: the slice's units shared evenly, or (whole) tiles of max_mu units in order, whose last one may reach
// past the slice.  Either way a row lies in one tile: two that both held it would both store it.
EIA_MOE_HD MoeTile moe_slice_tile(int rows, int tiles, int t, bool whole, int max_mu) {
  if (whole) return {max_mu * t, max_mu};
  const int units = (rows + 63) / 64, lo = units * t / tiles;
  return {lo, units * (t + 1) / tiles - lo};
}
