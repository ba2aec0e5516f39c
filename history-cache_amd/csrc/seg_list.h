// Lists of the long segments of an offsets array (rows of a CSR block, sources of a transposed view).
//
// A compute unit keeps about 85 cache lines in flight (measured, profiles/hbm_ceilings.md), so one that
// sums a segment of thousands of rows by itself takes a microsecond per 85 lines whatever its waves do:
// 0.9 ms for 10 000 rows of 1 KiB.  The long segments are therefore found first, by a launch that reads the
// offsets once, and the first blocks of the summing launch share them out: a task is one SLICE of columns
// (one cache line wide) of one segment, and consecutive tasks go to different compute units.
//
// The array is cut into at most SEG_MAX_REGIONS tiles, one block each.  A tile's part of a list starts at
// (entries in front of the tile) / (threshold + 1): the segments above the threshold in a tile are at most
// (entries of the tile) / (threshold + 1), so the parts cannot overlap, and neither a counter that has to be
// cleared nor a scan is needed.  The readers add up the (at most 512) counts themselves, eight per lane.
#pragma once

#include "hc_common.h"

constexpr int SEG_MAX_REGIONS = 512;

struct SegList {
  int32_t *count;   // per tile
  int32_t *item;    // segment numbers, part of tile t from seg_part(t) on
  int64_t cap;      // entries of `item`
};

// A wave's view of the counts: lane l holds the counts of tiles 8 l .. 8 l + 7.
struct SegIndex {
  int c[8];
  int incl;         // inclusive scan over the lanes
  int total;
};

__device__ __forceinline__ SegIndex seg_index(const int32_t *__restrict__ count, int n_tiles, int lane) {
  SegIndex x;
  int sum = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int r = lane * 8 + k;
    x.c[k] = r < n_tiles ? count[r] : 0;
    sum += x.c[k];
  }
  x.incl = sum;
#pragma unroll
  for (int d = 1; d < HC_WAVE; d <<= 1) {
    const int y = __shfl_up(x.incl, d, HC_WAVE);
    if (lane >= d) x.incl += y;
  }
  x.total = __builtin_amdgcn_readlane(x.incl, HC_WAVE - 1);
  return x;
}

// Tile and place inside its part of list entry e (wave-uniform, e < total).
__device__ __forceinline__ void seg_locate(const SegIndex &x, int e, int *tile, int *within) {
  const int l = __builtin_ctzll(__ballot(x.incl > e));
  int rem = e - (l > 0 ? __builtin_amdgcn_readlane(x.incl, l - 1) : 0);
  int k = 0;
#pragma unroll
  for (int i = 0; i < 7; ++i) {
    const int c = __builtin_amdgcn_readlane(x.c[i], l);
    if (k == i && rem >= c) {
      rem -= c;
      k = i + 1;
    }
  }
  *tile = l * 8 + k;
  *within = rem;
}

// Segments per tile: at least 1 024, few enough tiles for the readers.
inline int64_t seg_tile(int64_t n) {
  int64_t t = (n + SEG_MAX_REGIONS - 1) / SEG_MAX_REGIONS;
  t = (t + HC_BLOCK - 1) / HC_BLOCK * HC_BLOCK;
  return t < 1024 ? 1024 : t;
}

// Start of tile t's part of a list of the segments with more than `above` entries.
__device__ __forceinline__ int64_t seg_part(const int64_t *__restrict__ ptr, int64_t first, int64_t above) {
  return (ptr[first] - ptr[0]) / (above + 1);
}
