// Transposed (CSC) view of a CSR block, built with a stable sort so that the
// backward pass can gather instead of scattering with float atomics.
//
// The reference has no such step: its backward pushes gradients with
// atomicAdd (/root/reference/src/cpp/src/history_aggr.cu:164), which makes the
// sums depend on scheduling.  Here every source's incoming edges end up in
// ascending destination-row order, so the backward sums have one fixed order.
//
// Pipeline (all on the caller's stream):
//   1. expand    thread per edge slot: keys[e] = idx[e] and the slot's destination row (found by
//                binary search over the row offsets of the block's tile); slots outside the first R
//                rows and rows flagged by hmap_row get the sentinel key n_src
//   2. sort      rocPRIM LSD radix sort of (key, value) pairs -- stable.  When the caller wants
//                edgeT the value is the edge slot and rowT is gathered afterwards; when it does not
//                (mean aggregation) the value is the destination row and the sort writes rowT itself
//   3. finalize  ptrT[s] = first sorted position whose key is >= s
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "hc_common.h"
#include "tr_shared.h"

namespace {

// Sort input for every edge slot, one thread per slot: key = source id, or the sentinel for slots
// outside the first R rows, rows flagged by hmap_row and ids outside [0, n_src); value = edge slot
// (VAL_IS_ROW false; `rows[e]` then gets the destination row) or the destination row itself (mean
// aggregation; dropped slots carry their slot number, they sort behind every real key).
// A block covers TR_TILE consecutive slots.  The rows that overlap the tile are found with two
// binary searches; their offsets are staged in LDS when they fit, and every thread then finds the
// row of its slot with a short search.  Reads and writes are coalesced whatever the degrees are.
constexpr int TR_LDS_ROWS = 2048;
// slots per thread: 8 on large blocks; 1 on small ones (sampled batches), where more, shorter blocks
// matter more than the amortised tile search
constexpr int64_t TR_SORT_MEMSET_EDGES = 1 << 20;  // rocPRIM sorts up to this many pairs by merging (kernels only)
constexpr int TR_ITEMS_LARGE = 8;
constexpr int64_t TR_SMALL_EDGES = 1 << 18;

template <bool VAL_IS_ROW, int TR_ITEMS>
__global__ __launch_bounds__(HC_BLOCK) void tr_expand_edges(const int64_t *__restrict__ ptr,
                                                             const int64_t *__restrict__ idx,
                                                             const int64_t *__restrict__ hmap_row,
                                                             const int64_t *__restrict__ hmap_src,
                                                             const uint32_t *__restrict__ src_bits,
                                                             uint32_t *__restrict__ keys,
                                                             uint32_t *__restrict__ vals,
                                                             uint32_t *__restrict__ rows, int64_t R, int64_t E,
                                                             int64_t n_src) {
  constexpr int TR_TILE = HC_BLOCK * TR_ITEMS;
  __shared__ int64_t s_ptr[TR_LDS_ROWS];
  __shared__ int64_t s_range[2];
  const int64_t e0 = (int64_t)blockIdx.x * TR_TILE;
  const int64_t e1 = e0 + TR_TILE < E ? e0 + TR_TILE : E;
  if (threadIdx.x < 2 * HC_WAVE) {       // the tile's first and last row, searched by two waves side by side
    const int lane0 = hc_lane();
    const int which = (int)(threadIdx.x >> 6);
    const int64_t r = tr_row_of_wave(ptr, R, which == 0 ? e0 : e1 - 1, lane0);
    if (lane0 == 0) s_range[which] = r;
  }
  __syncthreads();
  const int64_t r_lo = s_range[0], r_hi = s_range[1];
  const int64_t span = r_hi - r_lo + 1;  // rows r_lo..r_hi (r_hi may be R: slots behind the last row)
  const bool staged = span <= TR_LDS_ROWS;
  if (staged)
    for (int64_t i = threadIdx.x; i < span; i += HC_BLOCK) s_ptr[i] = ptr[r_lo + i];
  __syncthreads();
  const uint32_t sentinel = (uint32_t)n_src;
  // three sweeps over the thread's slots, so that the loads of each sweep are all in flight together
  int64_t row[TR_ITEMS];
  bool live[TR_ITEMS];
#pragma unroll
  for (int it = 0; it < TR_ITEMS; ++it) {
    const int64_t e = e0 + (int64_t)it * HC_BLOCK + threadIdx.x;
    live[it] = false;
    row[it] = 0;
    if (e < e1) {
      if (staged) {
        const int64_t l = tr_row_of(s_ptr, (int64_t)0, span - 1, e);
        row[it] = r_lo + l;
        live[it] = row[it] < R && s_ptr[l] <= e;  // ptr[row + 1] > e by construction when row < R
      } else {
        row[it] = tr_row_of(ptr, r_lo, r_hi, e);
        live[it] = row[it] < R && ptr[row[it]] <= e;
      }
    }
  }
  if (hmap_row != nullptr) {
    int64_t h[TR_ITEMS];
#pragma unroll
    for (int it = 0; it < TR_ITEMS; ++it) h[it] = live[it] ? hmap_row[row[it]] : -1;
#pragma unroll
    for (int it = 0; it < TR_ITEMS; ++it) live[it] = live[it] && h[it] == -1;
  }
  int64_t src[TR_ITEMS];
#pragma unroll
  for (int it = 0; it < TR_ITEMS; ++it) {
    const int64_t e = e0 + (int64_t)it * HC_BLOCK + threadIdx.x;
    src[it] = live[it] ? idx[e] : -1;
  }
  if (hmap_src != nullptr) {   // sources that were substituted in the forward pass receive no gradient
    // src_bits (one bit per source, derived from the map by tr_src_bits) answers the question without
    // touching the map, which costs a cache line per lookup when the sources are many
    bool sub[TR_ITEMS];
#pragma unroll
    for (int it = 0; it < TR_ITEMS; ++it) {
      sub[it] = false;
      if (src[it] >= 0 && src[it] < n_src)
        sub[it] = src_bits != nullptr ? ((src_bits[src[it] >> 5] >> (src[it] & 31)) & 1u) != 0u
                                      : hmap_src[src[it]] != -1;
    }
#pragma unroll
    for (int it = 0; it < TR_ITEMS; ++it)
      if (sub[it]) {
        src[it] = -1;
        live[it] = false;
      }
  }
#pragma unroll
  for (int it = 0; it < TR_ITEMS; ++it) {
    const int64_t e = e0 + (int64_t)it * HC_BLOCK + threadIdx.x;
    if (e >= e1) continue;
    keys[e] = (src[it] >= 0 && src[it] < n_src) ? (uint32_t)src[it] : sentinel;
    if (VAL_IS_ROW) {
      vals[e] = live[it] ? (uint32_t)row[it] : (uint32_t)e;
    } else {
      vals[e] = (uint32_t)e;
      if (live[it]) rows[e] = (uint32_t)row[it];
    }
  }
}

__global__ __launch_bounds__(HC_BLOCK) void tr_finalize_edges(const uint32_t *__restrict__ skeys,
                                                               const uint32_t *__restrict__ svals,
                                                               const uint32_t *__restrict__ rows,
                                                               int32_t *__restrict__ rowT,
                                                               int32_t *__restrict__ edgeT, int64_t E,
                                                               uint32_t sentinel) {
  const int64_t p = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (p >= E) return;
  const uint32_t k = skeys[p];
  const uint32_t e = svals[p];
  if (k != sentinel) {
    rowT[p] = (int32_t)rows[e];
    edgeT[p] = (int32_t)e;
  } else {
    rowT[p] = -1;
    edgeT[p] = -1;
  }
}

// ptrT from the sorted keys by boundary detection: position p owns the sources in
// (key[p-1], key[p]] and writes ptrT[s] = p for them; the last position also closes the tail.
// Short runs are written by the owning lane; a long run (many consecutive sources without edges)
// is written by the whole wave, 64 entries per step, so no single lane loops for long.
__global__ __launch_bounds__(HC_BLOCK) void tr_ptr_from_boundaries(const uint32_t *__restrict__ skeys,
                                                                    int64_t *__restrict__ ptrT, int64_t E,
                                                                    int64_t n_src) {
  const int lane = hc_lane();
  const int64_t p = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  int64_t first = 0, last = -1;  // sources [first, last] get ptrT = p
  int64_t tail_first = 0, tail_last = -1;
  if (p < E) {
    const int64_t cur = skeys[p];
    const int64_t prev = p == 0 ? -1 : (int64_t)skeys[p - 1];
    first = prev + 1;
    last = cur;
    if (p == E - 1) {
      tail_first = cur + 1;
      tail_last = n_src;
    }
  }
  constexpr int64_t SHORT_RUN = 4;
  const int64_t run = last - first + 1;
  if (run > 0 && run <= SHORT_RUN)
    for (int64_t s = first; s <= last; ++s) ptrT[s] = p;
  // long runs: one at a time, by the whole wave
  unsigned long long m = __ballot(run > SHORT_RUN);
  while (m != 0ull) {
    const int l = __builtin_ctzll(m);
    m &= m - 1ull;
    const int64_t f = hc_readlane64(first, l);
    const int64_t t = hc_readlane64(last, l);
    const int64_t v = hc_readlane64(p, l);
    for (int64_t s = f + lane; s <= t; s += HC_WAVE) ptrT[s] = v;
  }
  // the tail behind the last key (at most one lane of the grid has one)
  unsigned long long mt = __ballot(tail_last >= tail_first);
  while (mt != 0ull) {
    const int l = __builtin_ctzll(mt);
    mt &= mt - 1ull;
    const int64_t f = hc_readlane64(tail_first, l);
    const int64_t t = hc_readlane64(tail_last, l);
    for (int64_t s = f + lane; s <= t; s += HC_WAVE) ptrT[s] = E;
  }
}

// ptrT[s] = number of sorted keys strictly below s, for s in [0, n_src] (binary search; used
// when there are many more sources than edges).
__global__ __launch_bounds__(HC_BLOCK) void tr_finalize_ptr(const uint32_t *__restrict__ skeys,
                                                             int64_t *__restrict__ ptrT, int64_t E,
                                                             int64_t n_src) {
  const int64_t s = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (s > n_src) return;
  int64_t lo = 0, hi = E;
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if ((int64_t)skeys[mid] < s) lo = mid + 1;
    else hi = mid;
  }
  ptrT[s] = lo;
}

// ---------------------------------------------------------------------------------------
// Small blocks (sampled mini-batches: at most TR_SMALL_EDGES edge slots and TR_SMALL_SOURCES sources):
// a counting sort in a few launches of this file's own kernels instead of the library sort's dozen.
//   tr_small_clear  zero the per-source counters
//   tr_small_count  thread per edge slot: the slot's key (source id, or the sentinel for a dropped
//                   slot) and destination row are saved and the source's counter is bumped (integer
//                   atomics: the final counts do not depend on their order)
//   tr_small_sums   (more than TRS_DIRECT_TILES tiles of 4096 sources) every tile's sum
//   tr_small_scan   block per tile: the counters become ptrT (exclusive scan) and per-source cursors; the
//                   sum in front of the tile is added up from the tiles' sums, or from the counters
//                   themselves where the tiles are few.  (One block that scanned all counters behind a
//                   ticket took 100 us of a batch of 230 000 sources; the two launches take 9.)
//   tr_small_place  thread per edge slot: takes the next free position of its source's segment
//                   (atomic: WHICH slots a segment holds is fixed, their order inside it is not yet)
//                   and writes (row, slot) there, into temporary arrays
//   tr_small_order  copies every segment to its final place in ascending slot order -- the order a
//                   stable sort gives: one-edge segments as they are, segments of up to 8 edges
//                   sorted by their lane in registers, of up to 64 edges ranked inside a wave, longer
//                   ones by the whole block through a bitmap of the segment's slots in LDS (rank =
//                   number of set bits below the slot), one window of TR_SMALL_EDGES slots at a time
// The result is bit-identical to the sorted view of the large-block path.
// The same kernels serve hc_build_transpose_dev, where the block's sizes are read from device
// memory (TrDims) and the launches are sized by capacities of up to 2^24 edge slots / sources.
// ---------------------------------------------------------------------------------------
constexpr int TRS_BLOCK = 1024;
constexpr int64_t TR_SMALL_SOURCES = 1 << 20;
constexpr int TRS_BITMAP_WORDS = (int)(TR_SMALL_EDGES / 32);   // one bit per edge slot
constexpr int TRS_ORDER_SOURCES = HC_BLOCK;                     // sources per block of tr_small_order
constexpr int TRS_LANE_SORT = 8;                                // longest segment a single lane sorts

constexpr int TRS_TILE = TRS_BLOCK * 4;                         // counters per block of the scan
constexpr int64_t TRS_DIRECT_TILES = 8;                         // up to so many tiles go without their sums

// Sizes of the block: given by value, or -- when the host does not know them yet (a batch that the
// sampler has just drawn) -- read from device memory and clamped to the bounds the launch was sized for.
struct TrDims {
  int64_t R, E, n_src;               // by value (or the upper bounds when the pointers are set)
  const int64_t *pR, *pE, *pS;       // nullable, all three or none
  int32_t *overflow;                 // nullable: set to 1 when a size read on the device had to be clamped, else 0
  int64_t *max_count;                // nullable: receives the largest number of live edges of one source
};
__device__ __forceinline__ void tr_dims(const TrDims &d, int64_t &R, int64_t &E, int64_t &n_src) {
  R = d.R;
  E = d.E;
  n_src = d.n_src;
  if (d.pE != nullptr) {
    const int64_t r = *d.pR, e = *d.pE, s = *d.pS;
    R = r < 0 ? 0 : r;               // rows are bounded by the caller's ptr array
    E = e < 0 ? 0 : (e < d.E ? e : d.E);
    n_src = s < 0 ? 0 : (s < d.n_src ? s : d.n_src);
  }
}
// Did tr_dims clamp anything?  (A view of a truncated block is a valid view of the wrong block.)
__device__ __forceinline__ bool tr_dims_clamped(const TrDims &d) {
  if (d.pE == nullptr) return false;
  const int64_t r = *d.pR, e = *d.pE, s = *d.pS;
  return r < 0 || e < 0 || s < 0 || e > d.E || s > d.n_src;
}

// zero the counters of sources [0, n_src] (rounded up to whole 16-byte groups)
__global__ __launch_bounds__(HC_BLOCK) void tr_small_clear(uint32_t *__restrict__ p, TrDims dims) {
  int64_t R, E, n_src;
  tr_dims(dims, R, E, n_src);
  const int64_t n = (n_src + 1 + 3) / 4 * 4;
  const int64_t i = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (i < n) p[i] = 0u;
  if (i == 0 && dims.overflow != nullptr) *dims.overflow = tr_dims_clamped(dims) ? 1 : 0;
  if (i == 0 && dims.max_count != nullptr) *dims.max_count = 0;
}

__global__ __launch_bounds__(TRS_BLOCK) void tr_small_count(
    const int64_t *__restrict__ ptr, const int64_t *__restrict__ idx, const int64_t *__restrict__ hmap_row,
    const int64_t *__restrict__ hmap_src, uint32_t *__restrict__ keys, int32_t *__restrict__ rows,
    int *__restrict__ count, TrDims dims) {
  __shared__ int64_t s_ptr[TR_LDS_ROWS];
  __shared__ int64_t s_range[2];
  int64_t R, E, n_src;
  tr_dims(dims, R, E, n_src);
  const int64_t e0 = (int64_t)blockIdx.x * TRS_BLOCK;
  const int64_t e1 = e0 + TRS_BLOCK < E ? e0 + TRS_BLOCK : E;
  if (e0 < E && R > 0) {                 // block-uniform (the launch may be sized for more edge slots)
    if (threadIdx.x < 2 * HC_WAVE) {       // the tile's first and last row, searched by two waves side by side
      const int lane0 = hc_lane();
      const int which = (int)(threadIdx.x >> 6);
      const int64_t r = tr_row_of_wave(ptr, R, which == 0 ? e0 : e1 - 1, lane0);
      if (lane0 == 0) s_range[which] = r;
    }
    __syncthreads();
    const int64_t r_lo = s_range[0], r_hi = s_range[1];
    const int64_t span = r_hi - r_lo + 1;
    const bool staged = span <= TR_LDS_ROWS;
    if (staged)
      for (int64_t i = threadIdx.x; i < span; i += TRS_BLOCK) s_ptr[i] = ptr[r_lo + i];
    __syncthreads();
    const int64_t e = e0 + threadIdx.x;
    if (e < e1) {
      int64_t row;
      bool live;
      if (staged) {
        const int64_t l = tr_row_of(s_ptr, (int64_t)0, span - 1, e);
        row = r_lo + l;
        live = row < R && s_ptr[l] <= e;
      } else {
        row = tr_row_of(ptr, r_lo, r_hi, e);
        live = row < R && ptr[row] <= e;
      }
      if (live && hmap_row != nullptr) live = hmap_row[row] == -1;
      int64_t src = live ? idx[e] : -1;
      if (src < 0 || src >= n_src) live = false;
      if (live && hmap_src != nullptr) live = hmap_src[src] == -1;
      keys[e] = live ? (uint32_t)src : (uint32_t)n_src;
      rows[e] = live ? (int32_t)row : -1;
      if (live) atomicAdd(count + src, 1);
    }
  }
}

// Four counters per thread.  Entries between n_src and the end of the counter array are zero.
__device__ __forceinline__ int4 trs_counters(const int *__restrict__ count, int64_t i, int64_t n_entries) {
  return i < (n_entries + 3) / 4 * 4 ? *reinterpret_cast<const int4 *>(count + i) : make_int4(0, 0, 0, 0);
}

// Sum over the block (every thread calls it; `s_wave` is free again when it returns).
__device__ __forceinline__ int trs_block_sum(int v, int *s_wave) {
#pragma unroll
  for (int d = HC_WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, HC_WAVE);
  if (hc_lane() == 0) s_wave[threadIdx.x >> 6] = v;
  __syncthreads();
  int sum = 0;
#pragma unroll
  for (int w = 0; w < TRS_BLOCK / HC_WAVE; ++w) sum += s_wave[w];
  __syncthreads();
  return sum;
}

__global__ __launch_bounds__(TRS_BLOCK) void tr_small_sums(const int *__restrict__ count, int *__restrict__ sums,
                                                            TrDims dims) {
  __shared__ int s_wave[TRS_BLOCK / HC_WAVE];
  int64_t R, E, n_src;
  tr_dims(dims, R, E, n_src);
  const int64_t base = (int64_t)blockIdx.x * TRS_TILE;
  if (base > n_src) return;
  const int4 c = trs_counters(count, base + (int64_t)threadIdx.x * 4, n_src + 1);
  const int sum = trs_block_sum((c.x + c.y) + (c.z + c.w), s_wave);
  if (threadIdx.x == 0) sums[blockIdx.x] = sum;
}

// `sums` nullable: the counters in front of the tile are added up here, while other blocks write their cursors (an
// array of its own).
__global__ __launch_bounds__(TRS_BLOCK) void tr_small_scan(const int *__restrict__ count, const int *__restrict__ sums,
                                                            int *__restrict__ cursor, int64_t *__restrict__ ptrT,
                                                            TrDims dims) {
  __shared__ int s_wave[TRS_BLOCK / HC_WAVE];
  int64_t R, E, n_src;
  tr_dims(dims, R, E, n_src);
  const int64_t base = (int64_t)blockIdx.x * TRS_TILE;
  const int64_t n_entries = n_src + 1;                      // ptrT has n_src + 1 entries
  if (base >= n_entries) return;
  const int lane = hc_lane();
  const int wave = (int)(threadIdx.x >> 6);
  const int64_t i = base + (int64_t)threadIdx.x * 4;
  const int4 c = trs_counters(count, i, n_entries);
  int before = 0;
  if (sums != nullptr) {
    for (int64_t t = threadIdx.x; t < (int64_t)blockIdx.x; t += TRS_BLOCK) before += sums[t];
  } else {
    for (int64_t t = 0; t < (int64_t)blockIdx.x; ++t) {
      const int4 p = trs_counters(count, t * TRS_TILE + (int64_t)threadIdx.x * 4, n_entries);
      before += (p.x + p.y) + (p.z + p.w);
    }
  }
  before = trs_block_sum(before, s_wave);
  const int mine = (c.x + c.y) + (c.z + c.w);
  int x = mine;                                             // inclusive scan over the wave
#pragma unroll
  for (int d = 1; d < HC_WAVE; d <<= 1) {
    const int y = __shfl_up(x, d, HC_WAVE);
    if (lane >= d) x += y;
  }
  if (lane == HC_WAVE - 1) s_wave[wave] = x;
  __syncthreads();
  int p0 = before + x - mine;
  for (int w = 0; w < wave; ++w) p0 += s_wave[w];
  const int p[4] = {p0, p0 + c.x, p0 + c.x + c.y, p0 + c.x + c.y + c.z};
  if (i + 3 < n_entries && reinterpret_cast<uintptr_t>(ptrT) % 16 == 0) {
    *reinterpret_cast<int4 *>(cursor + i) = make_int4(p[0], p[1], p[2], p[3]);      // the segments' cursors
    *reinterpret_cast<longlong2 *>(ptrT + i) = make_longlong2(p[0], p[1]);
    *reinterpret_cast<longlong2 *>(ptrT + i + 2) = make_longlong2(p[2], p[3]);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (i + j < n_entries) {
        cursor[i + j] = p[j];
        ptrT[i + j] = p[j];
      }
  }
  if (dims.max_count != nullptr) {                          // (kernel argument: the whole block takes the branch)
    int longest = max(max(c.x, c.y), max(c.z, c.w));
#pragma unroll
    for (int d = HC_WAVE / 2; d > 0; d >>= 1) longest = max(longest, __shfl_xor(longest, d, HC_WAVE));
    __syncthreads();                                        // s_wave is free again
    if (lane == 0) s_wave[wave] = longest;
    __syncthreads();
    if (threadIdx.x == 0) {                                 // one atomic per block: they queue at one address
      for (int w = 1; w < TRS_BLOCK / HC_WAVE; ++w) longest = max(longest, s_wave[w]);
      if (longest > 0) atomicMax(reinterpret_cast<unsigned long long *>(dims.max_count), (unsigned long long)longest);
    }
  }
}

__global__ __launch_bounds__(HC_BLOCK) void tr_small_place(const uint32_t *__restrict__ keys,
                                                            const int32_t *__restrict__ rows,
                                                            int *__restrict__ cursor,
                                                            int32_t *__restrict__ tmp_row,
                                                            int32_t *__restrict__ tmp_edge, TrDims dims) {
  int64_t R, E, n_src;
  tr_dims(dims, R, E, n_src);
  const int64_t e = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (e >= E || R <= 0) return;
  const uint32_t k = keys[e];
  if (k == (uint32_t)n_src) return;      // the sentinel of a dropped slot
  const int p = atomicAdd(cursor + k, 1);
  tmp_row[p] = rows[e];
  tmp_edge[p] = (int32_t)e;
}

__global__ __launch_bounds__(HC_BLOCK) void tr_small_order(const int64_t *__restrict__ ptrT,
                                                            const int32_t *__restrict__ tmp_row,
                                                            const int32_t *__restrict__ tmp_edge,
                                                            int32_t *__restrict__ rowT,
                                                            int32_t *__restrict__ edgeT, TrDims dims) {
  int64_t R_unused, E, n_src;
  tr_dims(dims, R_unused, E, n_src);
  __shared__ uint32_t bits[TRS_BITMAP_WORDS];
  __shared__ int pre8[TRS_BITMAP_WORDS / 8];
  __shared__ int long_src[TRS_ORDER_SOURCES];
  __shared__ int n_long_s;
  __shared__ int s_wave[HC_WAVES_PER_BLOCK];
  const int lane = hc_lane();
  const int wave = hc_wave_in_block();
  if (threadIdx.x == 0) n_long_s = 0;
  __syncthreads();
  // Popular sources tend to be neighbours (a sampled batch numbers them early), and a block works through its
  // long segments one after the other: the sources are dealt to the blocks eight at a time (a line of ptrT).
  const int64_t blocks = (n_src + TRS_ORDER_SOURCES - 1) / TRS_ORDER_SOURCES;
  if ((int64_t)blockIdx.x >= blocks) return;
  const auto source_of = [&](int t) -> int64_t { return ((int64_t)(t >> 3) * blocks + blockIdx.x) * 8 + (t & 7); };
  const int64_t s = source_of((int)threadIdx.x);
  int64_t b = 0;
  int len = 0;
  if (s < n_src) {
    b = ptrT[s];
    len = (int)(ptrT[s + 1] - b);
  }
  if (len == 1) {
    rowT[b] = tmp_row[b];
    if (edgeT != nullptr) edgeT[b] = tmp_edge[b];
  }
  if (len > HC_WAVE) long_src[atomicAdd(&n_long_s, 1)] = (int)threadIdx.x;
  // segments of 2..TRS_LANE_SORT edges (most of what is not a single edge): every lane sorts its own
  // segment in registers -- an odd-even transposition network on the slots, the rows ride along
  if (len >= 2 && len <= TRS_LANE_SORT) {
    int ve[TRS_LANE_SORT], vr[TRS_LANE_SORT];
#pragma unroll
    for (int k = 0; k < TRS_LANE_SORT; ++k) {
      ve[k] = k < len ? tmp_edge[b + k] : 0x7fffffff;
      vr[k] = k < len ? tmp_row[b + k] : 0;
    }
#pragma unroll
    for (int round = 0; round < TRS_LANE_SORT; ++round) {
#pragma unroll
      for (int k = round & 1; k + 1 < TRS_LANE_SORT; k += 2) {
        const bool sw = ve[k + 1] < ve[k];
        const int e0 = sw ? ve[k + 1] : ve[k], e1 = sw ? ve[k] : ve[k + 1];
        const int r0 = sw ? vr[k + 1] : vr[k], r1 = sw ? vr[k] : vr[k + 1];
        ve[k] = e0; ve[k + 1] = e1;
        vr[k] = r0; vr[k + 1] = r1;
      }
    }
#pragma unroll
    for (int k = 0; k < TRS_LANE_SORT; ++k) {
      if (k < len) {
        rowT[b + k] = vr[k];
        if (edgeT != nullptr) edgeT[b + k] = ve[k];
      }
    }
  }
  // segments of up to 64 edges: ranked inside the wave, one segment at a time
  unsigned long long m = __ballot(len > TRS_LANE_SORT && len <= HC_WAVE);
  while (m != 0ull) {
    const int l = __builtin_ctzll(m);
    m &= m - 1ull;
    const int64_t sb = hc_readlane64(b, l);
    const int sl = __builtin_amdgcn_readlane(len, l);
    const bool have = lane < sl;
    const int ve = have ? tmp_edge[sb + lane] : 0x7fffffff;
    const int vr = have ? tmp_row[sb + lane] : 0;
    int rank = 0;
    for (int j = 0; j < sl; ++j) rank += __builtin_amdgcn_readlane(ve, j) < ve ? 1 : 0;   // slots are distinct
    if (have) {
      rowT[sb + rank] = vr;
      if (edgeT != nullptr) edgeT[sb + rank] = ve;
    }
  }
  __syncthreads();
  // longer segments: the whole block, one segment at a time.  The segment's slots set their bits in an
  // LDS bitmap over a window of TR_SMALL_EDGES edge slots (one window covers a whole block of that size;
  // larger blocks take several); a slot's rank is the number of the segment's slots in earlier windows
  // plus the set bits below it in its own.
  const int n_long = n_long_s;
  for (int t = 0; t < n_long; ++t) {
    const int64_t src = source_of(long_src[t]);
    const int64_t sb = ptrT[src];
    const int sl = (int)(ptrT[src + 1] - sb);
    int before = 0;                                  // the segment's slots in the windows already done
    for (int64_t w0 = 0; w0 < E; w0 += TR_SMALL_EDGES) {
      const int64_t span = E - w0 < TR_SMALL_EDGES ? E - w0 : TR_SMALL_EDGES;
      const int words = (int)((span + 31) / 32);
      for (int w = threadIdx.x; w < words; w += HC_BLOCK) bits[w] = 0u;
      __syncthreads();
      for (int i = threadIdx.x; i < sl; i += HC_BLOCK) {
        const int64_t e = (int64_t)tmp_edge[sb + i] - w0;
        if (e >= 0 && e < span) atomicOr(&bits[e >> 5], 1u << (e & 31));
      }
      __syncthreads();
      // pre8[g] = set bits in front of word group g (8 words): per-thread run of groups, block scan
      const int groups = (words + 7) / 8;
      const int per = (groups + HC_BLOCK - 1) / HC_BLOCK;
      int glo = (int)threadIdx.x * per, ghi = glo + per;
      if (glo > groups) glo = groups;
      if (ghi > groups) ghi = groups;
      int sum = 0;
      for (int g = glo; g < ghi; ++g)
        for (int w = g * 8; w < g * 8 + 8 && w < words; ++w) sum += __popc(bits[w]);
      int x = sum;
#pragma unroll
      for (int d = 1; d < HC_WAVE; d <<= 1) {
        const int y = __shfl_up(x, d, HC_WAVE);
        if (lane >= d) x += y;
      }
      if (lane == HC_WAVE - 1) s_wave[wave] = x;
      __syncthreads();
      int run = before + x - sum;
      int in_window = 0;
      for (int w = 0; w < HC_WAVES_PER_BLOCK; ++w) {
        if (w < wave) run += s_wave[w];
        in_window += s_wave[w];
      }
      for (int g = glo; g < ghi; ++g) {
        pre8[g] = run;
        for (int w = g * 8; w < g * 8 + 8 && w < words; ++w) run += __popc(bits[w]);
      }
      __syncthreads();
      for (int i = threadIdx.x; i < sl; i += HC_BLOCK) {
        const int e_abs = tmp_edge[sb + i];
        const int64_t e = (int64_t)e_abs - w0;
        if (e < 0 || e >= span) continue;
        const int r = tmp_row[sb + i];
        const int w = (int)(e >> 5);
        int rank = pre8[w >> 3];
        for (int q = (w >> 3) * 8; q < w; ++q) rank += __popc(bits[q]);
        rank += __popc(bits[w] & ((1u << (e & 31)) - 1u));
        rowT[sb + rank] = r;
        if (edgeT != nullptr) edgeT[sb + rank] = e_abs;
      }
      before += in_window;
      __syncthreads();
    }
  }
}

struct SmallLayout {
  size_t count, cursor, sums, keys, rows, tmp_row, tmp_edge, total;
};
SmallLayout small_layout(int64_t E, int64_t n_src) {
  SmallLayout L;
  const size_t arr = hc_align_up((size_t)(E > 0 ? E : 1) * sizeof(uint32_t), 256);
  const size_t per_source = hc_align_up((size_t)(n_src + 1) * sizeof(int), 256);
  L.count = 0;
  L.cursor = per_source;
  L.sums = 2 * per_source;
  L.keys = L.sums + hc_align_up((size_t)(n_src / TRS_TILE + 1) * sizeof(int), 256);
  L.rows = L.keys + arr;
  L.tmp_row = L.rows + arr;
  L.tmp_edge = L.tmp_row + arr;
  L.total = L.tmp_edge + arr;
  return L;
}
inline bool small_block(int64_t E, int64_t n_src) { return E <= TR_SMALL_EDGES && n_src <= TR_SMALL_SOURCES; }
// Few edges over more sources than the small path takes: the library sorts them in one or two blocks, while the bucket
// sort's passes over a thousand buckets cost the same for any number of edges (us, library / buckets: 1000 edges over
// 2 M sources 24 / 50, over 5 M 38 / 46, over 20 M 104 / 98; 10 000 edges over 1.1 M 41 / 43, over 5 M 66 / 51).  Above
// 22 M sources the buckets' counters fill a compute unit's LDS (1000 edges over 40 M: 192 / 243).
constexpr int64_t TR_FEW_EDGES = 1 << 13;
constexpr int64_t TR_FEW_PRODUCT = (int64_t)1 << 34;
constexpr int64_t TR_WIDE_SOURCES = 22'000'000;
inline bool few_edges(int64_t E, int64_t n_src) {
  return E <= TR_FEW_EDGES && (E * n_src <= TR_FEW_PRODUCT || n_src > TR_WIDE_SOURCES);
}
// Larger blocks go to the bucket sort of view_sort.hip; what it does not cover (more than 2^28 edge slots or
// about 44 M sources) stays with the library sort below.  (Between 2^18 and 2^20 edges the library merges in a
// dozen launches: 600 k edges 150 us, 66 us with the bucket sort.)
inline bool bucket_sorted(int64_t E, int64_t n_src) {
  return !small_block(E, n_src) && !few_edges(E, n_src) && vs_supported(E, n_src);
}

// The launches of the counting sort; dims.E / dims.n_src size the grids (upper bounds when the real
// sizes are read on the device).
int small_launch(const int64_t *ptr, const int64_t *idx, const int64_t *hmap_row, const int64_t *hmap_src,
                 const TrDims &dims, int64_t *ptrT, int32_t *rowT, int32_t *edgeT, char *w, const SmallLayout &S,
                 hipStream_t st) {
  int *count = reinterpret_cast<int *>(w + S.count);
  int *cursor = reinterpret_cast<int *>(w + S.cursor);
  int *sums = reinterpret_cast<int *>(w + S.sums);
  uint32_t *keys = reinterpret_cast<uint32_t *>(w + S.keys);
  int32_t *rows = reinterpret_cast<int32_t *>(w + S.rows);
  int32_t *tmp_row = reinterpret_cast<int32_t *>(w + S.tmp_row);
  int32_t *tmp_edge = reinterpret_cast<int32_t *>(w + S.tmp_edge);
  const int64_t E = dims.E > 0 ? dims.E : 1, n_src = dims.n_src;
  const int64_t clear_words = (int64_t)(S.cursor / sizeof(uint32_t));
  const int64_t tiles = n_src / TRS_TILE + 1;
  const int64_t cb = (clear_words + HC_BLOCK - 1) / HC_BLOCK, eb = (E + TRS_BLOCK - 1) / TRS_BLOCK;
  const int64_t pb = (E + HC_BLOCK - 1) / HC_BLOCK, ob = (n_src + TRS_ORDER_SOURCES - 1) / TRS_ORDER_SOURCES;
  if (!hc_grid_ok(cb) || !hc_grid_ok(eb) || !hc_grid_ok(pb) || !hc_grid_ok(ob)) return HC_EUNSUPPORTED;
  tr_small_clear<<<dim3((unsigned)cb), dim3(HC_BLOCK), 0, st>>>(reinterpret_cast<uint32_t *>(count), dims);
  tr_small_count<<<dim3((unsigned)eb), dim3(TRS_BLOCK), 0, st>>>(ptr, idx, hmap_row, hmap_src, keys, rows, count, dims);
  if (tiles > TRS_DIRECT_TILES) tr_small_sums<<<dim3((unsigned)tiles), dim3(TRS_BLOCK), 0, st>>>(count, sums, dims);
  tr_small_scan<<<dim3((unsigned)tiles), dim3(TRS_BLOCK), 0, st>>>(count, tiles > TRS_DIRECT_TILES ? sums : nullptr, cursor,
                                                                   ptrT, dims);
  tr_small_place<<<dim3((unsigned)pb), dim3(HC_BLOCK), 0, st>>>(keys, rows, cursor, tmp_row, tmp_edge, dims);
  if (n_src > 0)
    tr_small_order<<<dim3((unsigned)ob), dim3(HC_BLOCK), 0, st>>>(ptrT, tmp_row, tmp_edge, rowT, edgeT, dims);
  return hc_launch_status();
}

// bits[s] = (hmap_src[s] != -1), 64 sources per ballot
__global__ __launch_bounds__(HC_BLOCK) void tr_src_bits(const int64_t *__restrict__ hmap, int64_t n_src,
                                                         unsigned long long *__restrict__ bits) {
  const int lane = hc_lane();
  const int64_t stride = (int64_t)gridDim.x * HC_WAVES_PER_BLOCK * HC_WAVE;
  for (int64_t base = ((int64_t)blockIdx.x * HC_WAVES_PER_BLOCK + hc_wave_in_block()) * HC_WAVE; base < n_src;
       base += stride) {
    const bool has = base + lane < n_src && hmap[base + lane] != -1;
    const unsigned long long bal = __ballot(has);
    if (lane == 0) bits[base / HC_WAVE] = bal;
  }
}

int key_bits(int64_t n_src) {
  int b = 1;
  while (b < 32 && ((int64_t)1 << b) <= n_src) ++b;
  return b;
}

struct Layout {
  size_t keys0, keys1, vals0, vals1, rows, bits, temp, total;
};

// The library's radix sort with the digit width and tile sizes chosen on this GPU: 9-bit digits (source
// ids of 19 to 27 bits take three passes instead of three to four 8-bit ones), 1024-thread blocks with 8
// keys per thread in the scatter kernel and 16 in the histogram kernel, wave-level ranking.  20 M pairs
// with 24-bit / 25-bit keys: 0.43 ms against 0.53 / 0.68 ms with the library's own choice; nine other
// combinations of digit width (8 - 11) and tile shape were slower.  Blocks below the merge-sort limit
// (2^20 pairs) are not affected.
using TrSortConfig = rocprim::radix_sort_config<
    rocprim::default_config, rocprim::default_config,
    rocprim::radix_sort_onesweep_config<rocprim::kernel_config<1024, 16>, rocprim::kernel_config<1024, 8>, 9,
                                        rocprim::block_radix_rank_algorithm::match>>;

hipError_t sort_temp_bytes(int64_t E, int bits, size_t *bytes) {
  rocprim::double_buffer<uint32_t> k(nullptr, nullptr), v(nullptr, nullptr);
  *bytes = 0;
  return rocprim::radix_sort_pairs<TrSortConfig>(nullptr, *bytes, k, v, (size_t)E, 0u, (unsigned)bits,
                                   (hipStream_t)0, false);
}

bool make_layout(int64_t E, int64_t n_src, Layout *L) {
  size_t temp = 0;
  if (E > 0 && sort_temp_bytes(E, key_bits(n_src), &temp) != hipSuccess) return false;
  const size_t arr = hc_align_up((size_t)(E > 0 ? E : 1) * sizeof(uint32_t), 256);
  L->keys0 = 0;
  L->keys1 = arr;
  L->vals0 = 2 * arr;
  L->vals1 = 3 * arr;
  L->rows = 4 * arr;
  L->bits = 5 * arr;   // one bit per source (used when a source map is given)
  L->temp = L->bits + hc_align_up((size_t)((n_src + 63) / 64) * 8 + 8, 256);
  L->total = L->temp + hc_align_up(temp > 0 ? temp : 1, 256);
  return true;
}

}  // namespace

extern "C" size_t hc_transpose_workspace_bytes(int64_t R, int64_t E, int64_t n_src) {
  (void)R;
  if (E < 0 || n_src < 0) return 0;
  if (small_block(E, n_src)) return small_layout(E, n_src).total;   // no library query on this path
  if (bucket_sorted(E, n_src)) return vs_workspace_bytes(E, n_src);
  Layout L;
  if (!make_layout(E, n_src, &L)) return 0;
  return L.total;
}

extern "C" int hc_build_transpose(const int64_t *ptr, const int64_t *idx, const int64_t *hmap_row,
                                  const int64_t *hmap_src, int64_t R, int64_t E, int64_t n_src, int64_t *ptrT,
                                  int32_t *rowT, int32_t *edgeT, void *workspace, size_t workspace_bytes,
                                  void *stream) {
  HC_REQUIRE(R >= 0 && E >= 0 && n_src >= 0 && ptrT);
  const int64_t lim = 0x7ffffffeLL;
  if (R > lim || E > lim || n_src > lim) return HC_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t pblocks = (n_src + 1 + HC_BLOCK - 1) / HC_BLOCK;
  if (E == 0 || R == 0) {
    // no edges: every segment is empty (binary search over zero keys writes 0)
    tr_finalize_ptr<<<dim3((unsigned)pblocks), dim3(HC_BLOCK), 0, st>>>(nullptr, ptrT, 0, n_src);
    return hc_launch_status();
  }
  HC_REQUIRE(ptr && idx && rowT);
  if (small_block(E, n_src)) {
    const SmallLayout S = small_layout(E, n_src);
    if (!workspace || workspace_bytes < S.total) return HC_EWORKSPACE;
    char *w = static_cast<char *>(workspace);
    if (reinterpret_cast<uintptr_t>(w) % 256 != 0) return HC_EWORKSPACE;
    const TrDims dims{R, E, n_src, nullptr, nullptr, nullptr, nullptr, nullptr};
    return small_launch(ptr, idx, hmap_row, hmap_src, dims, ptrT, rowT, edgeT, w, S, st);
  }
  if (bucket_sorted(E, n_src)) {
    char *w = static_cast<char *>(workspace);
    if (!workspace || reinterpret_cast<uintptr_t>(w) % 256 != 0) return HC_EWORKSPACE;
    return vs_launch(ptr, idx, hmap_row, hmap_src, R, E, n_src, ptrT, rowT, edgeT, w, workspace_bytes, st);
  }
  if (E > TR_SORT_MEMSET_EDGES) {
    // Above this size the sort library takes its one-sweep path, which clears its counters with
    // hipMemsetAsync; a captured graph would replay those as memset nodes.  Refuse instead.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(st, &cs) != hipSuccess) {
      (void)hipGetLastError();
    } else if (cs != hipStreamCaptureStatusNone) {
      return HC_EUNSUPPORTED;
    }
  }
  Layout L;
  if (!make_layout(E, n_src, &L)) return HC_ELAUNCH;
  if (!workspace || workspace_bytes < L.total) return HC_EWORKSPACE;
  char *ws = static_cast<char *>(workspace);
  if (reinterpret_cast<uintptr_t>(ws) % 256 != 0) return HC_EWORKSPACE;
  uint32_t *keys0 = reinterpret_cast<uint32_t *>(ws + L.keys0);
  uint32_t *keys1 = reinterpret_cast<uint32_t *>(ws + L.keys1);
  uint32_t *vals0 = reinterpret_cast<uint32_t *>(ws + L.vals0);
  uint32_t *vals1 = reinterpret_cast<uint32_t *>(ws + L.vals1);
  uint32_t *rows = reinterpret_cast<uint32_t *>(ws + L.rows);
  void *temp = ws + L.temp;
  size_t temp_bytes = L.total - L.temp;
  const uint32_t sentinel = (uint32_t)n_src;
  const uint32_t *src_bits = nullptr;
  if (hmap_src != nullptr && n_src >= ((int64_t)1 << 20)) {
    unsigned long long *bits = reinterpret_cast<unsigned long long *>(ws + L.bits);
    tr_src_bits<<<dim3(2048), dim3(HC_BLOCK), 0, st>>>(hmap_src, n_src, bits);
    src_bits = reinterpret_cast<const uint32_t *>(bits);
  }

  const int64_t eblocks = (E + HC_BLOCK - 1) / HC_BLOCK;
  const int64_t rblocks = (R + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
  if (!hc_grid_ok(eblocks) || !hc_grid_ok(rblocks) || !hc_grid_ok(pblocks)) return HC_EUNSUPPORTED;

  const bool want_edges = edgeT != nullptr;
  const unsigned bits = (unsigned)key_bits(n_src);
  const uint32_t *skeys = nullptr;
  const int items = E <= TR_SMALL_EDGES ? 1 : TR_ITEMS_LARGE;
  const int64_t tile = (int64_t)HC_BLOCK * items;
  const dim3 tgrid((unsigned)((E + tile - 1) / tile));
  if (want_edges) {
    if (items == 1)
      tr_expand_edges<false, 1><<<tgrid, dim3(HC_BLOCK), 0, st>>>(ptr, idx, hmap_row, hmap_src, src_bits, keys0, vals0, rows, R, E, n_src);
    else
      tr_expand_edges<false, TR_ITEMS_LARGE><<<tgrid, dim3(HC_BLOCK), 0, st>>>(ptr, idx, hmap_row, hmap_src, src_bits, keys0,
                                                                               vals0, rows, R, E, n_src);
    rocprim::double_buffer<uint32_t> dk(keys0, keys1), dv(vals0, vals1);
    if (rocprim::radix_sort_pairs<TrSortConfig>(temp, temp_bytes, dk, dv, (size_t)E, 0u, bits, st, false) != hipSuccess)
      return HC_ELAUNCH;
    tr_finalize_edges<<<dim3((unsigned)eblocks), dim3(HC_BLOCK), 0, st>>>(dk.current(), dv.current(), rows,
                                                                          rowT, edgeT, E, sentinel);
    skeys = dk.current();
  } else {
    // value = destination row; dropped edge slots keep the fill value and sort behind the sentinel
    if (items == 1)
      tr_expand_edges<true, 1><<<tgrid, dim3(HC_BLOCK), 0, st>>>(ptr, idx, hmap_row, hmap_src, src_bits, keys0, vals0, nullptr, R, E, n_src);
    else
      tr_expand_edges<true, TR_ITEMS_LARGE><<<tgrid, dim3(HC_BLOCK), 0, st>>>(ptr, idx, hmap_row, hmap_src, src_bits, keys0,
                                                                              vals0, nullptr, R, E, n_src);
    // rowT doubles as the sort's second value buffer; copy only if the result landed in the first
    uint32_t *rowT_u = reinterpret_cast<uint32_t *>(rowT);
    rocprim::double_buffer<uint32_t> dk(keys0, keys1), dv(vals0, rowT_u);
    if (rocprim::radix_sort_pairs<TrSortConfig>(temp, temp_bytes, dk, dv, (size_t)E, 0u, bits, st, false) != hipSuccess)
      return HC_ELAUNCH;
    if (dv.current() != rowT_u &&
        hipMemcpyAsync(rowT, dv.current(), (size_t)E * sizeof(uint32_t), hipMemcpyDeviceToDevice, st) != hipSuccess)
      return HC_ELAUNCH;
    skeys = dk.current();
  }
  if (n_src <= 4 * E) {
    tr_ptr_from_boundaries<<<dim3((unsigned)eblocks), dim3(HC_BLOCK), 0, st>>>(skeys, ptrT, E, n_src);
  } else {
    tr_finalize_ptr<<<dim3((unsigned)pblocks), dim3(HC_BLOCK), 0, st>>>(skeys, ptrT, E, n_src);
  }
  return hc_launch_status();
}

// Limits of the variant with device-resident sizes: the counters are 32-bit and one block scans them.
constexpr int64_t TR_DEV_MAX_EDGES = (int64_t)1 << 24;
constexpr int64_t TR_DEV_MAX_SOURCES = (int64_t)1 << 24;

extern "C" size_t hc_transpose_dev_workspace_bytes(int64_t max_E, int64_t max_src) {
  if (max_E < 0 || max_src < 0 || max_E > TR_DEV_MAX_EDGES || max_src > TR_DEV_MAX_SOURCES) return 0;
  return small_layout(max_E, max_src).total;
}

extern "C" int hc_build_transpose_dev(const int64_t *ptr, const int64_t *idx, const int64_t *R_dev,
                                      const int64_t *E_dev, const int64_t *n_src_dev, int64_t max_E,
                                      int64_t max_src, int64_t *ptrT, int32_t *rowT, int32_t *edgeT,
                                      int32_t *overflow, void *workspace, size_t workspace_bytes, void *stream) {
  return hc_build_transpose_dev_deg(ptr, idx, R_dev, E_dev, n_src_dev, max_E, max_src, ptrT, rowT, edgeT, overflow,
                                    nullptr, workspace, workspace_bytes, stream);
}

extern "C" int hc_build_transpose_dev_deg(const int64_t *ptr, const int64_t *idx, const int64_t *R_dev,
                                          const int64_t *E_dev, const int64_t *n_src_dev, int64_t max_E,
                                          int64_t max_src, int64_t *ptrT, int32_t *rowT, int32_t *edgeT,
                                          int32_t *overflow, int64_t *max_in_degree, void *workspace,
                                          size_t workspace_bytes, void *stream) {
  HC_REQUIRE(ptr && idx && R_dev && E_dev && n_src_dev && ptrT && max_E >= 0 && max_src >= 0);
  HC_REQUIRE(rowT != nullptr || max_E == 0);
  if (max_E > TR_DEV_MAX_EDGES || max_src > TR_DEV_MAX_SOURCES) return HC_EUNSUPPORTED;
  const SmallLayout S = small_layout(max_E, max_src);
  if (!workspace || workspace_bytes < S.total) return HC_EWORKSPACE;
  char *w = static_cast<char *>(workspace);
  if (reinterpret_cast<uintptr_t>(w) % 256 != 0) return HC_EWORKSPACE;
  const TrDims dims{0, max_E, max_src, R_dev, E_dev, n_src_dev, overflow, max_in_degree};
  return small_launch(ptr, idx, nullptr, nullptr, dims, ptrT, rowT, edgeT, w, S, static_cast<hipStream_t>(stream));
}
