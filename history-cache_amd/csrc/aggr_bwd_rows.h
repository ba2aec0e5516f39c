// History-aware aggregation, backward, as a gather over the transposed view.
//
// Every SOURCE row s is summed in ascending destination-row order: g[r,:]/deg(r) (mean) or
// g[r,:]*edge_value[j] (weighted) over the edges that point at s.  No float atomics: each output
// element has one writer and a fixed summation order, the same order a sequential walk of the CSR
// block in row/edge order produces.
//
// Semantics follow the reference kernels gen_bwd_history_grad_v2*
// (/root/reference/src/cpp/src/history_aggr.cu:127-397): history rows route
// g[r,:] to grads_history[r,:] undivided (:144-149) and push nothing to their
// neighbours; the other rows push g/deg (:140-142,161-166) or g*edge_value
// (:209).
//
// A wave owns a run of consecutive sources.  Their incoming edges are one contiguous span of the transposed
// arrays, so the wave streams that span 64 edges at a time (one coalesced load of destination rows, one gather
// of their degrees) and walks it with a wave-uniform cursor: when the cursor passes the end of a source's
// segment the accumulator is stored (zeros for sources without edges) and reset.
//
// What bounds it: a large block of evenly used sources runs at the memory system's rate; a block with popular
// sources was bound by the waves that owned them, since popular sources tend to be neighbours (32 of them held
// 7 000 edges, a millisecond for one wave).  Two things share the work out:
//   * a run of sources ends where its edges plus four per source pass a multiple of BWD_UNIT (bwd_prepare
//     writes where each run starts), so that no wave owns more than 32 sources or about BWD_UNIT + BWD_LONG
//     edges;
//   * sources of more than BWD_LONG edges are listed by the same launch and summed by the front blocks of the
//     main one, a cache line's columns at a time (seg_list.h): 32 loads of one line in flight instead of eight
//     of whole rows, and one source on several compute units.
// Of a shared view's long sources the front blocks visit the live edges only (BwdLive): a layer of 50 rows over a view
// with sources of 10 000 edges takes 24 us (101 when every dead edge cost a load, 50 before there were lists).
// Measured on MI355X, before (fixed runs of 32 sources; widths off a multiple of 64 element by element; the
// conversion of a half-precision gradient as a pass of its own) and after, lists included: 3 M edges x 256 to
// 1 M bf16 sources 2.37 -> 0.38 ms, 1 M edges x 4 heads of 32 to 200 k sources 0.95 -> 0.08 ms, 600 k edges x 100
// 0.264 -> 0.055 ms, 10 k edges x 128 73 -> 25 us, 20 M edges x 256 to 10 M evenly used sources 3.28 -> 3.19 ms.
#pragma once

#include "hc_common.h"
#include "seg_list.h"

constexpr int BWD_XCD_CHUNK = 64;   // consecutive blocks that share an XCD
// The plain mean over a width of bwd_fast_shape, with a workspace: a source with more edges than this is summed
// in chunks of BWD_CHUNK edges, the chunk sums added left to right.
constexpr int BWD_CHUNK = 512;
constexpr int BWD_LONG = 128;       // sources with more edges are the front blocks' tasks
// A chunked source above this many edges is several blocks' work: each leaves its chunks' sums in the workspace and
// the one that arrives last adds them left to right.  (A compute unit brings in about 65 lines a microsecond, whatever
// its waves do.  4 M edges x 256 with a source of 1.0 M and 70 above 4 096: 3.5 ms by a wave per chunk, 1.2 ms so.)
constexpr int BWD_SPAN = 8 * BWD_CHUNK;
constexpr int BWD_UNIT = 128;       // a wave's run of sources: edges + BWD_SRC_COST per source
constexpr int BWD_SRC_COST = 4;
constexpr int BWD_MAX_RUN = 32;     // BWD_UNIT / BWD_SRC_COST; fixed runs have at most this many sources too
constexpr int BWD_FRONT_BLOCKS = 2048;
constexpr int W_NONE = 0, W_EDGE = 1, W_EDGE_HEAD = 2;

struct BwdArgs {
  const int64_t *ptr, *ptrT;
  const int32_t *rowT, *edgeT;
  const float *ev;
  int n_head;
  const float *g;
  const int64_t *hmap;
  void *grad_vin;
  float *grad_hbuf;             // nullable
  int64_t hsize;
  int64_t R, n_src;
  int64_t E;                    // entries of the view that the lists and the runs are sized for
  int64_t F;                    // a row is all heads side by side
  int slots;                    // F / VEC
  bool small_matrix;            // g holds less than 4 GiB
  int64_t long_above;           // sources with more edges are left to the front blocks (0: none)
  int64_t chunk;                // sources with more edges are summed in chunks (0: never); >= long_above
  SegList mid, hub, giant;      // long sources up to `chunk` (or all of them), up to BWD_SPAN, the others
  uint32_t *ticket;             // per giant and slice, zeroed by bwd_prepare
  int64_t n_tickets;
  float *partial;               // chunk sums of the giants, two rows per BWD_CHUNK positions of the view
  int n_tiles;
  int64_t tile;
  int front;
  const int32_t *run_start;     // nullable: first source of every run; else runs of `run` sources
  int32_t *run_start_out;
  int run;
  int64_t src_blocks, hist_blocks;
};

__device__ __forceinline__ int64_t bwd_run_of(const BwdArgs &a, int64_t s) {
  return (a.ptrT[s] + (int64_t)BWD_SRC_COST * s) / BWD_UNIT;
}

// v / d from r = 1 / d rounded once: the quotient's residual is exact in a fused multiply-add, and adding
// residual * r rounds to the quotient (Markstein, IBM J. Res. Dev. 34, 1990).  These are the division's bits where the
// quotient is normal and the whole divisor is below 2^22: such a quotient lies further from the rounding boundaries
// than the residual's error reaches.  A subnormal quotient that is an exact tie may become either of its two nearest
// neighbours (9 * 2^-149 / 6 the odd one), and above 2^22 one that close to a tie may; the error is no larger than a
// division's.  The fix-up passes infinities, NaN and signed zeros on as a division does.  Five instructions shorter
// than the division, which took more issue slots of a row than its loads.  (Looking every quotient over, to divide
// where it is subnormal: 14 M edges x 64 1.33 -> 1.39 ms, slices of a long source 104 -> 120 us.)
__device__ __forceinline__ float bwd_div(float v, float d, float r) {
  const float q = __fmul_rn(v, r);
  return __builtin_amdgcn_div_fixupf(__fmaf_rn(__fmaf_rn(-q, d, v), r, q), d, v);
}

// MASKED: the view covers the whole mini-batch CSR; transposed edges whose destination row lies outside
// the first R rows, took its history row (hmap[row] != -1), or is left empty by the layer's own offsets (a
// batch padded for a recorded iteration keeps the rows behind a layer's real ones empty, while the batch's shared
// view still lists their edges) are stepped over: row -1.
struct BwdEdge {
  int row;      // -1: stepped over
  float d, r;   // mean: the row's edges and their reciprocal; W_EDGE: d is the weight
  int edge;     // W_EDGE_HEAD: the edge's slot
};
template <int WMODE, bool MASKED>
__device__ __forceinline__ BwdEdge bwd_edge(const BwdArgs &a, int64_t pos, int row) {
  BwdEdge e{row, 1.0f, 1.0f, 0};
  if constexpr (MASKED) {
    if (row >= a.R || row < 0) e.row = -1;
    else if (a.hmap != nullptr && a.hmap[row] != -1) e.row = -1;
  }
  if constexpr (WMODE == W_EDGE_HEAD) {
    e.edge = a.edgeT[pos];
  } else if constexpr (WMODE == W_EDGE) {
    e.d = a.ev[a.edgeT[pos]];
  } else if (!MASKED || e.row >= 0) {
    e.d = (float)(int)(a.ptr[e.row + 1] - a.ptr[e.row]);
    if (MASKED && e.d == 0.0f) {
      e.row = -1;
      e.d = 1.0f;
    }
    e.r = 1.0f / e.d;
  }
  return e;
}

// Columns of a lane: chunk k holds elements off[k] .. off[k] + VEC - 1; lanes behind the row's end read
// the last slot again (no extra line) and store nothing.
template <int VEC, int CHUNKS>
struct BwdCols {
  uint32_t off[CHUNKS];
  bool on[CHUNKS];
  int hd[CHUNKS];
  __device__ __forceinline__ BwdCols(const BwdArgs &a, int tile, int lane, bool heads) {
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k) {
      const int slot = (tile * CHUNKS + k) * HC_WAVE + lane;
      on[k] = slot < a.slots;
      off[k] = (uint32_t)(on[k] ? slot : a.slots - 1) * VEC;
      hd[k] = heads ? (int)(off[k] / (uint32_t)(a.F / a.n_head)) : 0;
    }
  }
};

// Element c of a row of g (wave-uniform).
template <bool BUF>
__device__ __forceinline__ float bwd_element(const BwdArgs &a, hc_buffer buf, uint32_t row_bytes, int row, uint32_t c) {
  if constexpr (BUF) return __uint_as_float(hc_buffer_load<uint32_t>(buf, c * 4u, (uint32_t)row * row_bytes));
  else return __uint_as_float(hc_piece<float, 1>::template load<false>(reinterpret_cast<int64_t>(a.g + (int64_t)row * a.F), c * 4u));
}

// One column per lane of transposed edges [begin, end), added in edge order, D to 2 D gradient rows in flight:
// the loads of a group of D rows are issued before the adds of the group in front of it, the rows of the next 64
// edges at the start of this stage and their degrees or weights behind its first group.
// BUF: g is smaller than 4 GiB and its rows are addressed by 32-bit offsets from scalar registers.
template <int WMODE, bool BUF>
__device__ __forceinline__ float bwd_slice_sum(const BwdArgs &a, uint32_t c, int64_t begin, int64_t end, int lane) {
  constexpr int D = 16;
  constexpr int G = HC_WAVE / D;
  float acc = 0.0f;
  if (begin >= end) return acc;
  // several heads: the lanes of a slice may lie in different ones
  const int hd = WMODE == W_EDGE_HEAD ? (int)(c / (uint32_t)(a.F / a.n_head)) : 0;
  const hc_buffer buf = hc_make_buffer(a.g);
  const uint32_t row_bytes = (uint32_t)a.F * 4u;
  float x[2][D], w[2][WMODE == W_EDGE_HEAD ? D : 1];
  const auto load = [&](int h, const BwdEdge &e, int g, int last) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      int j = g * D + u;
      j = j < last ? j : last;                               // behind the end: the last row again, not added
      const int row = __builtin_amdgcn_readlane(e.row, j);
      x[h][u] = bwd_element<BUF>(a, buf, row_bytes, row, c);
      if constexpr (WMODE == W_EDGE_HEAD) w[h][u] = a.ev[(int64_t)__builtin_amdgcn_readlane(e.edge, j) * a.n_head + hd];
    }
  };
  const auto add1 = [&](int h, int u, const BwdEdge &e, int j) {
    if constexpr (WMODE == W_EDGE_HEAD) acc += __fmul_rn(x[h][u], w[h][u]);
    else if constexpr (WMODE == W_EDGE) acc += __fmul_rn(x[h][u], hc_readlane_f(e.d, j));
    else acc += bwd_div(x[h][u], hc_readlane_f(e.d, j), hc_readlane_f(e.r, j));
  };
  int64_t p = begin + lane < end ? begin + lane : end - 1;
  BwdEdge cur = bwd_edge<WMODE, false>(a, p, a.rowT[p]);
  int last = end - begin < HC_WAVE ? (int)(end - begin) - 1 : HC_WAVE - 1;
  load(0, cur, 0, last);
  int64_t base = begin;
  for (; base + HC_WAVE <= end; base += HC_WAVE) {
    const int64_t next = base + HC_WAVE;
    p = next + lane < end ? next + lane : end - 1;
    const int next_row = a.rowT[p];
    BwdEdge ahead = cur;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G) {
        load((g + 1) & 1, cur, g + 1, HC_WAVE - 1);
      } else {
        last = end - next < HC_WAVE ? (int)(end - next) - 1 : HC_WAVE - 1;
        load(0, ahead, 0, last < 0 ? 0 : last);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < D; ++u) add1(g & 1, u, cur, g * D + u);
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) ahead = bwd_edge<WMODE, false>(a, p, next_row);
    }
    cur = ahead;
  }
  // the last, partial stage: its first group is on its way
  const int n = (int)(end - base);
  for (int g = 0; g * D < n; ++g) {
    if (g > 0) load(0, cur, g, n - 1);
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (g * D + u < n) add1(0, u, cur, g * D + u);
  }
  return acc;
}

// The live edges of a stretch of a shared view, put together 64 at a time: BWD_WINDOWS windows of 64 positions are
// looked at together and the rows that are live go to a ring in the LDS.
constexpr int BWD_WINDOWS = 4, BWD_RING = 512;       // a ring holds what is left of a stage and all of the windows
struct BwdLive {
  int *ring;
  int64_t pos, end;                                  // next position to be looked at
  int head, count;
  int next[BWD_WINDOWS];                             // the rows from `pos` on, on their way
  __device__ __forceinline__ BwdLive(const BwdArgs &a, int *ring_, int64_t begin, int64_t end_, int lane)
      : ring(ring_), pos(begin), end(end_), head(0), count(0) {
    fetch(a, lane);
  }
  __device__ __forceinline__ void fetch(const BwdArgs &a, int lane) {
#pragma unroll
    for (int w = 0; w < BWD_WINDOWS; ++w) {
      const int64_t p = pos + w * HC_WAVE + lane;
      next[w] = a.rowT[p < end ? p : end - 1];
    }
  }
  // The next up to 64 live edges, in order; their number.  Lanes behind them hold the last one again.
  __device__ __forceinline__ int take(const BwdArgs &a, int lane, BwdEdge &e) {
    const unsigned long long below = (1ull << lane) - 1ull;
    while (count < HC_WAVE && pos < end) {           // wave-uniform
      int row[BWD_WINDOWS];
      bool live[BWD_WINDOWS];
      int64_t slot[BWD_WINDOWS];
#pragma unroll
      for (int w = 0; w < BWD_WINDOWS; ++w) {
        row[w] = next[w];
        live[w] = pos + w * HC_WAVE + lane < end && row[w] >= 0 && row[w] < a.R;
      }
      pos += BWD_WINDOWS * HC_WAVE;
      fetch(a, lane);
#pragma unroll
      for (int w = 0; w < BWD_WINDOWS; ++w) slot[w] = live[w] && a.hmap != nullptr ? a.hmap[row[w]] : -1;
#pragma unroll
      for (int w = 0; w < BWD_WINDOWS; ++w) {
        live[w] = live[w] && slot[w] == -1;
        const unsigned long long b = __ballot(live[w]);
        if (live[w]) ring[(head + count + __popcll(b & below)) % BWD_RING] = row[w];
        count += __popcll(b);
      }
    }
    const int n = count < HC_WAVE ? count : HC_WAVE;
    if (n == 0) return 0;
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");     // (the LDS serves a wave in order)
    e = BwdEdge{ring[(head + (lane < n ? lane : n - 1)) % BWD_RING], 1.0f, 1.0f, 0};
    head = (head + n) % BWD_RING;
    count -= n;
    e.d = (float)(int)(a.ptr[e.row + 1] - a.ptr[e.row]);
    if (e.d == 0.0f) {
      e.row = -1;
      e.d = 1.0f;
    }
    e.r = 1.0f / e.d;
    return n;
  }
};

// bwd_slice_sum of the mean over the live edges of a shared view.
template <bool BUF>
__device__ __forceinline__ float bwd_live_sum(const BwdArgs &a, uint32_t c, int64_t begin, int64_t end, int lane, int *ring) {
  constexpr int D = 16;
  constexpr int G = HC_WAVE / D;
  float acc = 0.0f;
  if (begin >= end) return acc;
  const hc_buffer buf = hc_make_buffer(a.g);
  const uint32_t row_bytes = (uint32_t)a.F * 4u;
  float x[2][D];
  const auto load = [&](int h, const BwdEdge &e, int g, int last) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      int j = g * D + u;
      j = j < last ? j : last;                               // behind the end: the last row again, not added
      const int row = __builtin_amdgcn_readlane(e.row, j);
      x[h][u] = bwd_element<BUF>(a, buf, row_bytes, row < 0 ? 0 : row, c);       // without edges of its own: not added
    }
  };
  const auto add1 = [&](int h, int u, const BwdEdge &e, int j) {
    const float q = bwd_div(x[h][u], hc_readlane_f(e.d, j), hc_readlane_f(e.r, j));
    acc += __builtin_amdgcn_readlane(e.row, j) < 0 ? 0.0f : q;                   // acc is never -0
  };
  BwdLive live(a, ring, begin, end, lane);
  BwdEdge cur{0, 1.0f, 1.0f, 0};
  int n = live.take(a, lane, cur);
  if (n > 0) load(0, cur, 0, n - 1);
  while (n == HC_WAVE) {
    BwdEdge ahead = cur;
    int m = 0;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G) load((g + 1) & 1, cur, g + 1, HC_WAVE - 1);
      else load(0, ahead, 0, m > 0 ? m - 1 : 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < D; ++u) add1(g & 1, u, cur, g * D + u);
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) m = live.take(a, lane, ahead);
    }
    cur = ahead;
    n = m;
  }
  for (int g = 0; g * D < n; ++g) {
    if (g > 0) load(0, cur, g, n - 1);
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (g * D + u < n) add1(0, u, cur, g * D + u);
  }
  return acc;
}

template <int WMODE, bool MASKED>
__device__ __forceinline__ float bwd_slice_any(const BwdArgs &a, uint32_t c, int64_t begin, int64_t end, int lane, int *ring) {
  if constexpr (MASKED)
    return a.small_matrix ? bwd_live_sum<true>(a, c, begin, end, lane, ring) : bwd_live_sum<false>(a, c, begin, end, lane, ring);
  else
    return a.small_matrix ? bwd_slice_sum<WMODE, true>(a, c, begin, end, lane) : bwd_slice_sum<WMODE, false>(a, c, begin, end, lane);
}

constexpr int BWD_SLICE = 32;       // columns of a task: one cache line of g

// The front blocks: a task is one slice of one listed source; a chunked source's slice is a block's task, whose
// waves sum a chunk each at a time, the others are a wave's.
template <typename TO, int WMODE, bool MASKED>
__device__ __forceinline__ void bwd_front(const BwdArgs &a, int lane, int wave) {
  __shared__ float part[HC_WAVES_PER_BLOCK][BWD_SLICE];
  __shared__ int rings[MASKED ? HC_WAVES_PER_BLOCK : 1][MASKED ? BWD_RING : 1];
  int *ring = rings[MASKED ? wave : 0];
  const int ns = (int)((a.F + BWD_SLICE - 1) / BWD_SLICE);
  const auto source = [&](const SegList &list, const SegIndex &index, int64_t above, int e) -> int64_t {
    int t, w;
    seg_locate(index, e, &t, &w);
    return (int64_t)__builtin_amdgcn_readfirstlane(list.item[seg_part(a.ptrT, (int64_t)t * a.tile, above) + w]);
  };
  // the lane's column of slice `sl`; lanes behind the slice or the row read its last one again
  const auto column = [&](int sl, bool &on) -> uint32_t {
    const int c = sl * BWD_SLICE + (lane < BWD_SLICE ? lane : BWD_SLICE - 1);
    on = lane < BWD_SLICE && c < a.F;
    return (uint32_t)(c < a.F ? c : a.F - 1);
  };
  TO *__restrict__ out = static_cast<TO *>(a.grad_vin);
  if (WMODE == W_NONE && a.giant.cap > 0) {
    __shared__ int s_last;
    const SegIndex index = seg_index(a.giant.count, a.n_tiles, lane);
    int64_t t = blockIdx.x;                                  // this block's next task, counted from the giant's first
    for (int i = 0; i < index.total; ++i) {                  // block-uniform
      const int64_t s = source(a.giant, index, BWD_SPAN, i);
      const int64_t b = a.ptrT[s], e = a.ptrT[s + 1];
      const int64_t spans = (e - b + BWD_SPAN - 1) / BWD_SPAN;
      // chunk k starts at position b + k * BWD_CHUNK; its window holds one other start at most, a first chunk's
      const auto row = [&](int64_t k) -> float * {
        return a.partial + (2 * ((b + k * BWD_CHUNK) / BWD_CHUNK) + (k == 0 ? 1 : 0)) * a.F;
      };
      for (; t < spans * ns; t += a.front) {
        const int sl = (int)(t % ns);
        bool on;
        const uint32_t c = column(sl, on);
        for (int64_t k = t / ns * (BWD_SPAN / BWD_CHUNK) + wave; k < (t / ns + 1) * (BWD_SPAN / BWD_CHUNK);
             k += HC_WAVES_PER_BLOCK) {
          const int64_t mb = b + k * BWD_CHUNK;
          if (mb >= e) break;
          const float v = bwd_slice_any<W_NONE, MASKED>(a, c, mb, mb + BWD_CHUNK < e ? mb + BWD_CHUNK : e, lane, ring);
          if (on) row(k)[c] = v;
        }
        if (hc_arrives_last(a.ticket + (int64_t)i * ns + sl, (unsigned)spans, &s_last)) {
          if (wave == 0) {
            const int64_t n = (e - b + BWD_CHUNK - 1) / BWD_CHUNK;
            float sum = row(0)[c];
            int64_t k = 1;
            for (; k + 8 <= n; k += 8) {
              float v[8];
#pragma unroll
              for (int u = 0; u < 8; ++u) v[u] = row(k + u)[c];
#pragma unroll
              for (int u = 0; u < 8; ++u) sum += v[u];
            }
            for (; k < n; ++k) sum += row(k)[c];
            if (on) out[s * a.F + c] = hc_from_f32<TO>(sum);
          }
        }
        __syncthreads();
      }
      t -= spans * ns;
    }
  }
  if (WMODE == W_NONE && a.chunk > 0) {
    const SegIndex index = seg_index(a.hub.count, a.n_tiles, lane);
    const int64_t tasks = (int64_t)index.total * ns;
    for (int64_t t = blockIdx.x; t < tasks; t += a.front) {
      const int64_t s = source(a.hub, index, a.chunk, (int)(t / ns));
      bool on;
      const uint32_t c = column((int)(t % ns), on);
      const int64_t b = a.ptrT[s], e = a.ptrT[s + 1];
      float sum = 0.0f;
      for (int64_t c0 = b; c0 < e; c0 += HC_WAVES_PER_BLOCK * BWD_CHUNK) {     // block-uniform
        const int64_t mb = c0 + wave * BWD_CHUNK < e ? c0 + wave * BWD_CHUNK : e;
        const int64_t me = mb + BWD_CHUNK < e ? mb + BWD_CHUNK : e;
        const float v = bwd_slice_any<W_NONE, MASKED>(a, c, mb, me, lane, ring);
        if (lane < BWD_SLICE) part[wave][lane] = v;
        __syncthreads();
        if (wave == 0 && lane < BWD_SLICE) {
#pragma unroll
          for (int w = 0; w < HC_WAVES_PER_BLOCK; ++w) {
            if (c0 == b && w == 0) sum = part[0][lane];
            else if (c0 + w * BWD_CHUNK < e) sum += part[w][lane];
          }
        }
        __syncthreads();
      }
      if (wave == 0 && on) out[s * a.F + c] = hc_from_f32<TO>(sum);
    }
  }
  const SegIndex index = seg_index(a.mid.count, a.n_tiles, lane);
  const int64_t tasks = (int64_t)index.total * ns;
  for (int64_t t = (int64_t)wave * a.front + blockIdx.x; t < tasks; t += (int64_t)HC_WAVES_PER_BLOCK * a.front) {
    const int64_t s = source(a.mid, index, a.long_above, (int)(t / ns));
    bool on;
    const uint32_t c = column((int)(t % ns), on);
    const float v = bwd_slice_any<WMODE, MASKED>(a, c, a.ptrT[s], a.ptrT[s + 1], lane, ring);
    if (on) out[s * a.F + c] = hc_from_f32<TO>(v);
  }
}

// WMODE W_EDGE: every transposed edge contributes g[row] * edge_value[edge] (product rounded, then
// added) instead of g[row] / deg(row); edgeT gives the edge slot of a transposed edge.
// WMODE W_EDGE_HEAD: a row is n_head heads side by side and the weight is edge_value[edge, head]; a
// lane's VEC elements of a chunk lie inside one head, whose weight the lane loads itself.  (grad_hbuf
// of such blocks is written by bwd_hist_generic.)
// TO: element type of grad_vin; the fp32 sums are rounded once when a source is stored.
// Blocks: front blocks, blocks of source runs, rows of grad_hbuf.
template <typename TO, int VEC, int CHUNKS, int UNROLL, int WMODE, bool MASKED>
__device__ __forceinline__ void bwd_block(const BwdArgs &a) {
  const int lane = hc_lane();
  const int wave = hc_wave_in_block();
  if ((int)blockIdx.x < a.front) {
    bwd_front<TO, WMODE, MASKED>(a, lane, wave);
    return;
  }
  const int64_t block = (int64_t)blockIdx.x - a.front;
  if (block >= a.src_blocks) {
    // grad_hbuf rows: copy g for history rows, zero otherwise
    const int64_t row = (block - a.src_blocks) * HC_WAVES_PER_BLOCK + wave;
    if (row >= a.R) return;
    const bool hit = a.hmap[row] != -1;
    float *__restrict__ d = a.grad_hbuf + row * a.hsize;
    const float *__restrict__ s = a.g + row * a.F;
    if (a.hsize == a.F && (reinterpret_cast<uintptr_t>(a.grad_hbuf) % 16) == 0) {
      for (int slot = lane; slot < a.slots; slot += HC_WAVE) {
        float v[VEC];
        if (hit) {
          hc_vec<float, VEC>::load(s + (int64_t)slot * VEC, v);
        } else {
#pragma unroll
          for (int i = 0; i < VEC; ++i) v[i] = 0.0f;
        }
        hc_vec<float, VEC>::store_nt(d + (int64_t)slot * VEC, v);
      }
      return;
    }
    for (int64_t c = lane; c < a.hsize; c += HC_WAVE) d[c] = (hit && c < a.F) ? s[c] : 0.0f;
    return;
  }
  const int64_t unit = hc_xcd_block<BWD_XCD_CHUNK>(block, a.src_blocks) * HC_WAVES_PER_BLOCK + wave;
  int64_t s0, s1;
  // every thread of the grid reads the same two words, so the decision is uniform: a view of more entries than its
  // caller announced is summed as if there were neither lists (bwd_prepare leaves them empty) nor runs, which would not
  // hold it
  const bool listed = a.front > 0 && a.ptrT[a.n_src] - a.ptrT[0] <= a.E;
  if (a.run_start != nullptr && listed) {
    const int64_t last = bwd_run_of(a, a.n_src);
    if (unit > last) return;
    s0 = a.run_start[unit];
    s1 = unit < last ? a.run_start[unit + 1] : a.n_src;
  } else {
    const int64_t run = a.run_start != nullptr ? BWD_MAX_RUN : a.run;      // the runs' waves are no fewer than those
    s0 = unit * run;
    s1 = s0 + run < a.n_src ? s0 + run : a.n_src;
  }
  s0 = hc_uniform64(s0);
  s1 = hc_uniform64(s1);
  if (s0 >= s1) return;
  const int ns = (int)(s1 - s0);                 // at most BWD_MAX_RUN
  // lane l holds the segment bound ptrT[s0 + l], l = 0..ns
  const int64_t my_p = a.ptrT[s0 + (lane < ns ? lane : ns)];
  const int64_t my_p1 = a.ptrT[s0 + (lane + 1 < ns ? lane + 1 : ns)];
  // sources summed by the front blocks: their segments are stepped over and not stored here
  const unsigned long long long_mask =
      listed ? __ballot(lane < ns && (my_p1 - my_p) > a.long_above) : 0ull;
  const int tiles = CHUNKS == 4 ? (a.slots + HC_WAVE * CHUNKS - 1) / (HC_WAVE * CHUNKS) : 1;
  for (int tile = 0; tile < tiles; ++tile) {
    const BwdCols<VEC, CHUNKS> col(a, tile, lane, WMODE == W_EDGE_HEAD);
    float acc[CHUNKS][VEC];
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[k][i] = 0.0f;
    int cur = 0;                                   // source (relative to s0) being accumulated
    int64_t cur_end = hc_readlane64(my_p, 1);      // end of its segment
    TO *__restrict__ obase = static_cast<TO *>(a.grad_vin) + s0 * a.F;
    int64_t base = hc_readlane64(my_p, 0);
    const auto store = [&]() {
#pragma unroll
      for (int k = 0; k < CHUNKS; ++k)
        if (col.on[k]) hc_vec<TO, VEC>::store_nt(obase + (int64_t)cur * a.F + col.off[k], acc[k]);
    };
    while (true) {  // every branch below advances `cur` or `base`; all of it is wave-uniform
      // close the sources whose segment ends at or before `base` (zeros for sources without edges)
      while (cur < ns && base >= cur_end) {
        if (((long_mask >> cur) & 1ull) == 0ull) store();
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
          for (int i = 0; i < VEC; ++i) acc[k][i] = 0.0f;
        ++cur;
        cur_end = hc_readlane64(my_p, cur + 1 <= ns ? cur + 1 : ns);
      }
      if (cur >= ns) break;
      if ((long_mask >> cur) & 1ull) {  // step over a long source's segment
        base = cur_end;
        continue;
      }
      // stage up to 64 edges, stopping in front of the next long source's segment
      const unsigned long long ahead = long_mask >> cur;
      const int nh = ahead != 0ull ? cur + __builtin_ctzll(ahead) : ns;
      const int64_t stop = hc_readlane64(my_p, nh);
      const int64_t left = stop - base;
      const int n = left < HC_WAVE ? (int)left : HC_WAVE;
      BwdEdge my{-1, 1.0f, 1.0f, 0};
      if (lane < n) my = bwd_edge<WMODE, MASKED>(a, base + lane, a.rowT[base + lane]);
      // MASKED: only the live edges of the stage are visited (lowest position first), so that UNROLL rows are
      // in flight however many edges of other layers lie between them
      unsigned long long todo = 0ull;
      if constexpr (MASKED) todo = __ballot(lane < n && my.row >= 0);
      for (int j = 0; MASKED ? todo != 0ull : j < n; j += UNROLL) {
        typename hc_piece<float, VEC>::raw_t v[UNROLL][CHUNKS];
        float d[UNROLL], r1[UNROLL];
        bool on[UNROLL];
        int pos[UNROLL];
        float wh[WMODE == W_EDGE_HEAD ? UNROLL : 1][CHUNKS];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          d[u] = r1[u] = 1.0f;
          if constexpr (MASKED) {
            on[u] = todo != 0ull;
            pos[u] = on[u] ? __builtin_ctzll(todo) : 0;
            todo &= todo - 1ull;                     // 0 stays 0
          } else {
            on[u] = j + u < n;
            pos[u] = j + u;
          }
          if (on[u]) {
            const int r = __builtin_amdgcn_readlane(my.row, pos[u]);
            if constexpr (WMODE != W_EDGE_HEAD) d[u] = hc_readlane_f(my.d, pos[u]);
            if constexpr (WMODE == W_NONE) r1[u] = hc_readlane_f(my.r, pos[u]);
            const int64_t p = reinterpret_cast<int64_t>(a.g + (int64_t)r * a.F);
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) v[u][k] = hc_piece<float, VEC>::template load<false>(p, col.off[k] * 4u);
            if constexpr (WMODE == W_EDGE_HEAD) {
              const int64_t e = (int64_t)__builtin_amdgcn_readlane(my.edge, pos[u]) * a.n_head;
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k) wh[u][k] = a.ev[e + col.hd[k]];
            }
          }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          if (on[u]) {
            const int64_t e = base + pos[u];
            while (e >= cur_end) {  // close finished (possibly empty) segments; none of them is a long one
              store();
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
                for (int i = 0; i < VEC; ++i) acc[k][i] = 0.0f;
              ++cur;
              cur_end = hc_readlane64(my_p, cur + 1);
            }
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
              for (int i = 0; i < VEC; ++i) {
                const float x = hc_piece<float, VEC>::widen(v[u][k], i);
                if constexpr (WMODE == W_EDGE_HEAD) acc[k][i] += __fmul_rn(x, wh[u][k]);
                else if constexpr (WMODE == W_EDGE) acc[k][i] += __fmul_rn(x, d[u]);
                else acc[k][i] += bwd_div(x, d[u], r1[u]);
              }
          }
        }
      }
      base += n;
    }
  }
}

// The mean: at most 80 scalar registers; above, fewer waves fit the chip (14 M edges x 64 1326 us, 1295 so).
template <typename TO, int VEC, int CHUNKS, int UNROLL>
__global__ __launch_bounds__(HC_BLOCK) __attribute__((amdgpu_num_sgpr(80))) void bwd_sources(BwdArgs a) {
  bwd_block<TO, VEC, CHUNKS, UNROLL, W_NONE, false>(a);
}

// Weights: what their slices take.
template <typename TO, int VEC, int CHUNKS, int UNROLL, int WMODE>
__global__ __launch_bounds__(HC_BLOCK) void bwd_sources_weighted(BwdArgs a) {
  bwd_block<TO, VEC, CHUNKS, UNROLL, WMODE, false>(a);
}

// The vector registers of the live edges' slices leave four waves per SIMD, whatever the scalar ones.
template <typename TO, int VEC, int CHUNKS, int UNROLL>
__global__ __launch_bounds__(HC_BLOCK) void bwd_sources_of_view(BwdArgs a) {
  bwd_block<TO, VEC, CHUNKS, UNROLL, W_NONE, true>(a);
}

// One translation unit per element type of grad_vin.
__attribute__((visibility("hidden"))) int bwd_dispatch_f32(BwdArgs &a, bool masked, hipStream_t st);
__attribute__((visibility("hidden"))) int bwd_dispatch_f16(BwdArgs &a, bool masked, hipStream_t st);
__attribute__((visibility("hidden"))) int bwd_dispatch_bf16(BwdArgs &a, bool masked, hipStream_t st);

#ifdef BWD_INSTANTIATE
namespace {

template <typename TO, int VEC, int CHUNKS>
int bwd_launch(const BwdArgs &a, bool masked, hipStream_t st) {
  constexpr int per = VEC * CHUNKS;
  constexpr int UNROLL = per >= 16 ? 4 : (per >= 4 ? 8 : 16);
  const int64_t blocks = a.front + a.src_blocks + a.hist_blocks;
  if (!hc_grid_ok(blocks)) return HC_EUNSUPPORTED;
  const dim3 grid((unsigned)blocks), block(HC_BLOCK);
  if (masked) bwd_sources_of_view<TO, VEC, CHUNKS, UNROLL><<<grid, block, 0, st>>>(a);
  else if (a.ev != nullptr && a.n_head > 1) bwd_sources_weighted<TO, VEC, CHUNKS, UNROLL, W_EDGE_HEAD><<<grid, block, 0, st>>>(a);
  else if (a.ev != nullptr) bwd_sources_weighted<TO, VEC, CHUNKS, UNROLL, W_EDGE><<<grid, block, 0, st>>>(a);
  else bwd_sources<TO, VEC, CHUNKS, UNROLL><<<grid, block, 0, st>>>(a);
  return hc_launch_status();
}

template <typename TO, int VEC>
int bwd_launch_chunks(const BwdArgs &a, bool masked, hipStream_t st) {
  const int chunks = (a.slots + HC_WAVE - 1) / HC_WAVE;
  if (chunks <= 1) return bwd_launch<TO, VEC, 1>(a, masked, st);
  if (chunks == 2) return bwd_launch<TO, VEC, 2>(a, masked, st);
  if (chunks == 3) return bwd_launch<TO, VEC, 3>(a, masked, st);
  return bwd_launch<TO, VEC, 4>(a, masked, st);         // wider rows: column tiles of 256 slots
}

// Elements per lane and load: the widest power of two that the row length, a head's width and the pointers
// allow, halved while the row still fits the wave.
template <typename TO>
int bwd_dispatch(BwdArgs &a, bool masked, hipStream_t st) {
  const int64_t fh = a.F / a.n_head;
  const auto fits = [&](int v) {
    return fh % v == 0 && reinterpret_cast<uintptr_t>(a.g) % (v * sizeof(float)) == 0 &&
           reinterpret_cast<uintptr_t>(a.grad_vin) % (v * sizeof(TO)) == 0;
  };
  int v = 4;
  while (v > 1 && (!fits(v) || a.F / (v / 2) <= HC_WAVE)) v /= 2;
  a.slots = (int)(a.F / v);
  if (v == 4) return bwd_launch_chunks<TO, 4>(a, masked, st);
  if (v == 2) return bwd_launch_chunks<TO, 2>(a, masked, st);
  return bwd_launch_chunks<TO, 1>(a, masked, st);
}

}  // namespace
#endif  // BWD_INSTANTIATE
