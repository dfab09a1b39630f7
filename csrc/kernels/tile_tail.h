// Which 256 x 256 tile of a dense or grouped product covers what, and which tiles are its tail.
#pragma once
#include <hip/hip_runtime.h>

#include "common.h"

#define TG_BM 256
#define TG_BN 256
#define TG_BAND 4
#define TG_CUS 256

// Tiles `cut` and up are cut in `splits` ranges of the reduction (1: none is).
struct TileTail {
  int cut, splits;
};

// A round is 256 workgroups, one a CU.  Its last round costs a product a whole tile's time however few tiles it has: up to half a round of
// them are cut so that they fill it.  A range costs what a whole tile does beside its chunks (about six chunks' time for its first loads and
// its 256 KiB of sums) and the tail a pass of 5 to 13 us, 4 to 9 chunks' time: fewer than six chunks a range are not worth it, nor a tail
// alone that saves fewer than 16 chunks.  Whole / cut, microseconds, the chunks saved in brackets: 512 x 6144, 24 chunks 39.9 / 35.0 (18), 250 x
// 1536, 23 chunks 31.6 / 27.2 (16); the last product and the sum of eight experts, hidden 2816, 400 tokens, 32 chunks 111 / 107 (16).  (Dense
// products whose ranges fill the round need 22, a pass of their own: ops/__init__.py.)  Behind whole
// rounds workgroups are out of step and part of the last one's time is hidden: 36 chunks (28672 x 4096 gated, 336 tiles, 43 saved 157 and 145;
// 896 tiles, 32 saved 341 and 341; 4096 x 4096, 384 tiles, 32 saved 196 and 206), and none behind eight and more (37888 x 3584, 3108 tiles 1063
// and 1089).
__host__ __device__ __forceinline__ TileTail tile_tail(int tiles, int chunks) {
  const int rest = tiles % TG_CUS;
  if (rest == 0 || rest > TG_CUS / 2 || tiles >= 8 * TG_CUS) return {tiles, 1};
  int s = TG_CUS / rest;
  if (s > chunks / 6) s = chunks / 6;
  if (s < 2 || chunks - chunks / s < (tiles < TG_CUS ? 16 : 36)) return {tiles, 1};
  return {tiles - rest, s};
}

struct TileAt {
  int group, row0, row_end, n_idx, units;
};

// Rows offsets[g] .. offsets[g + 1] of every group in tiles of up to 256 (offsets null: one group of max_rows), dealt out evenly in units of
// 64 (ragged) or in whole tiles.  Tile order: group by group; inside a group bands of TG_BAND column tiles; inside a band row tile by
// row tile.
struct TileRows {
  const int* offsets;
  int n_groups, max_rows, n_tiles;
  bool ragged;

  __device__ __forceinline__ static int m_tiles(int lo, int hi) { return (hi - lo + TG_BM - 1) / TG_BM; }
  __device__ __forceinline__ int tiles() const {
    if (!offsets) return m_tiles(0, max_rows) * n_tiles;
    int total = 0;
    for (int g = 0; g < n_groups; ++g) total += m_tiles(offsets[g], offsets[g + 1]) * n_tiles;
    return total;
  }
  // The same by a whole wave, a group a lane: of 32 experts, one after another takes 4 to 6 us of loads that wait for each other.
  __device__ __forceinline__ int tiles_by_wave() const {
    if (!offsets) return tiles();
    int mine = 0;
    for (int g = threadIdx.x & 63; g < n_groups; g += 64) mine += m_tiles(offsets[g], offsets[g + 1]);
    return __builtin_amdgcn_readfirstlane((int)wave_reduce_sum((float)mine)) * n_tiles;  // (whole below 2^24 row tiles)
  }
  // tile t of all
  __device__ __forceinline__ TileAt at(int t) const {
    TileAt r = {0, 0, 0, 0, 4};
    for (int first = 0; r.group < n_groups; ++r.group) {
      const int lo = offsets ? offsets[r.group] : 0, hi = offsets ? offsets[r.group + 1] : max_rows, m = m_tiles(lo, hi);
      if (t < first + m * n_tiles) {
        const int tl = t - first, per_band = m * TG_BAND, band = tl / per_band, rem = tl - band * per_band;
        const int width = (band + 1) * TG_BAND <= n_tiles ? TG_BAND : n_tiles - band * TG_BAND, m_idx = rem / width;
        r.n_idx = band * TG_BAND + (rem - m_idx * width);
        const int all = (hi - lo + 63) / 64, each = all / m, more = all - each * m;
        r.units = ragged ? each + (m_idx < more) : 4;
        r.row0 = ragged ? lo + 64 * (m_idx * each + (m_idx < more ? m_idx : more)) : lo + m_idx * TG_BM;
        r.row_end = hi;
        break;
      }
      first += m * n_tiles;
    }
    return r;
  }
  // the group of a row: its first tile and its rows
  __device__ __forceinline__ void group_of(int row, int& first, int& lo, int& hi) const {
    first = 0;
    for (int g = 0; g < n_groups; ++g) {
      lo = offsets[g];
      hi = offsets[g + 1];
      if (row < hi) return;
      first += m_tiles(lo, hi) * n_tiles;
    }
  }
  // a row of a group: its row tile and that tile's first row
  __device__ __forceinline__ void row_tile(int lo, int hi, int row, int& m_idx, int& row0) const {
    const int m = m_tiles(lo, hi), all = (hi - lo + 63) / 64, each = all / m, more = all - each * m, unit = (row - lo) / 64;
    if (!ragged) m_idx = (row - lo) / TG_BM;
    else m_idx = unit < more * (each + 1) ? unit / (each + 1) : more + (unit - more * (each + 1)) / each;
    row0 = lo + (ragged ? 64 * (m_idx * each + (m_idx < more ? m_idx : more)) : m_idx * TG_BM);
  }
  // a tile's place in its group
  __device__ __forceinline__ int tile_index(int m, int m_idx, int n_idx) const {
    const int band = n_idx / TG_BAND, width = (band + 1) * TG_BAND <= n_tiles ? TG_BAND : n_tiles - band * TG_BAND;
    return band * m * TG_BAND + m_idx * width + (n_idx - band * TG_BAND);
  }
};
