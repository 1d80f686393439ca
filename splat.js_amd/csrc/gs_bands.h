// gs_bands.h — into how many bands of tile rows the scatter of the
// tile-segment binning splits a view (gs_sort.hip).
//
// Each of an XCD's blocks fills one line of every tile's segment at a time;
// where those lines pass the XCD's 4 MB L2, each 8-byte key goes to memory as
// a partial write of its own, and the pass runs at that rate (77 Gkeys/s, as a
// bare kernel of such stores). So the blocks take the tiles in bands of rows
// whose open lines (128 bytes x blocks per XCD x tiles) stay within 3 MB, and
// walk their Gaussians once per band. 1920x1080, 1M Gaussians, 92.6M keys:
// 1156 us in one band, 694, 658 and 905 us in bands of 3, 6 and 12 rows (1.5,
// 2.9 and 5.9 MB).
//
// A band saves about 5 ps per key and costs a walk of all Gaussians, so it
// takes enough keys for both:
// - 12 per block and tile: at 44, 26, 15, 9 and 5 of them (1M Gaussians) the
//   bands take 660, 433, 329, 259 and 217 us against 1156, 680, 405, 249 and
//   162 without. Shorter runs of keys do not fill their lines either way.
// - 3 per band and Gaussian above 2^19 (few Gaussians stay in the L2s between
//   walks, and a walk of more reads them from memory, 14 ps each). The whole
//   binning at 1920x1080 (12 bands), without and with bands: 3M Gaussians with
//   30M, 56M, 93M and 157M keys 892 and 1276, 1551 and 1888, 2481 and 2594,
//   4234 and 3971 us; 10M with 35M, 65M, 117M and 188M 1252 and 2803, 1979 and
//   3450, 3268 and 4624, 5187 and 6341.
//
// Included from C (tests) and from HIP device code.
#ifndef GS_BANDS_H
#define GS_BANDS_H
#include <stdint.h>

#include "gs_math.h"

// tile rows per band for `keys` keys of n Gaussians, scattered by nb blocks
// into numTiles tiles, tilesX to a row; 0: one band (sparse views, most of
// them, leave before the first division: each costs a block some 20 cycles)
GS_HD int gs_band_rows(uint64_t keys, int64_t n, int nb, int tilesX, int numTiles) {
  const int lines = (3 << 20) / 128;   // open lines per XCD
  if (keys < (uint64_t)12 * (uint64_t)nb * (uint64_t)numTiles) return 0;
  const int tilesY = numTiles / tilesX, fit = lines / ((nb + 7) / 8) / tilesX, rows = fit < 1 ? 1 : fit;
  if (rows >= tilesY) return 0;
  const int64_t bands = (tilesY + rows - 1) / rows, walked = n - (1 << 19);
  return walked > 0 && keys < (uint64_t)(3 * bands * walked) ? 0 : rows;
}

#endif
