// History-aware CSR gather-reduce, forward.
//
// One wavefront owns one destination row.  The row's neighbour ids are staged
// 64 at a time with one coalesced load (one id per lane); each id is then
// broadcast with v_readlane so the neighbour row's base address is
// wave-uniform and the 64 lanes read one contiguous span of the row with
// vector loads (as wide as the row length and the pointers' alignment allow).
// Up to UNROLL neighbour rows are in flight per wave before the first add; the
// adds run in CSR order in fp32.  Rows of up to 256 edges are therefore summed in
// exactly the order a sequential CPU loop would use; longer rows (mean and
// single-head weights) are summed as four contiguous quarters combined left to
// right -- a fixed order, so results stay bit-reproducible.
//
// What bounds it: the bulk of a block is bound by the memory system (5 - 6 TB/s of random rows once the chip is
// full), the rest by its longest rows, which are therefore shared out slice by slice (seg_list.h).  Measured on
// MI355X, before (rows of four waves, widths off a multiple of 64 element by element) and after: 3 M edges x 256
// bf16 with a row of 14 000 edges 1.42 -> 0.26 ms; 600 k edges x 100 fp32 0.64 -> 0.047 ms; 20 M edges x 256 fp32
// over 20 GB 4.20 -> 4.20 ms (its long rows are short beside the launch).
//
// Semantics follow the reference kernels gen_fwd_history_v2,
// gen_fwd_history_v2_edge_value and gen_fwd_history_v2_edge_value_multi_head
// (/root/reference/src/cpp/src/history_aggr.cu:7-125); offsets are 64-bit
// (the reference truncates neighbour ids and offsets to 32-bit int, :19,34-35).
#pragma once

#include "hc_common.h"
#include "seg_list.h"

#include <type_traits>
#include <utility>

// Rows with more edges than this are summed as four quarters (mean, single-head weights).
// The oracle applies the same rule; the header documents it.
constexpr int64_t HC_LONG_ROW_EDGES = 256;
// Rows of several heads are never split into quarters; those above this many edges are summed slice by
// slice on several compute units (each slice strictly in CSR order).
constexpr int64_t FWD_HEAD_SLICE_EDGES = 128;

// Wave-cooperative copy of one row of a history buffer into an fp32 output row.
template <typename TH>
__device__ __forceinline__ void copy_row_typed(const TH *__restrict__ src, float *__restrict__ dst,
                                               int64_t F, int lane) {
  constexpr int V = 4;
  const bool vec_ok = (F % V == 0) && ((reinterpret_cast<uintptr_t>(src) % (sizeof(TH) * V)) == 0) &&
                      ((reinterpret_cast<uintptr_t>(dst) % 16) == 0);
  if (vec_ok) {
    for (int64_t c = (int64_t)lane * V; c < F; c += HC_WAVE * V) {
      float v[V];
      hc_vec<TH, V>::load(src + c, v);
      *reinterpret_cast<float4 *>(dst + c) = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else {
    for (int64_t c = lane; c < F; c += HC_WAVE) dst[c] = hc_to_f32<TH>(src[c]);
  }
}

__device__ __forceinline__ void copy_row_any(const void *hbuf, int hist_dtype, int64_t elem_off,
                                             float *dst, int64_t F, int lane) {
  if (hist_dtype == HC_F32) {
    copy_row_typed<float>(static_cast<const float *>(hbuf) + elem_off, dst, F, lane);
  } else if (hist_dtype == HC_F16) {
    copy_row_typed<__half>(static_cast<const __half *>(hbuf) + elem_off, dst, F, lane);
  } else {
    copy_row_typed<__hip_bfloat16>(static_cast<const __hip_bfloat16 *>(hbuf) + elem_off, dst, F, lane);
  }
}

// WMODE 0: acc += row.  WMODE 1: acc = fma(row, edge_value[edge], acc).  WMODE 2: the row holds
// n_head heads side by side and every head has its own weight, edge_value[edge, head]; a lane's VEC
// elements of a chunk lie inside one head, whose weight the lane loads itself.
constexpr int W_NONE = 0, W_EDGE = 1, W_EDGE_HEAD = 2;

// What the main launch does with the lists.  (Worked out by each of its waves, with two 64-bit divisions, it took 1 M
// rows of 3 edges of 64 columns from 443 to 526 us.)
struct FwdPlan {
  int64_t far_above, listed, staged_above;
  int64_t staged, staged_fit;  // with staged rows, written by fwd_stage: rows in staged_order, and how many of them have copies
};

// Rows of several heads are never split: the longest of them is one chain of additions, and a wave that follows it
// through the matrix gets 64 lines a microsecond.  Where such a row takes longer than everything else in the launch, a
// launch of its own copies its source rows side by side first (fwd_stage), in slices of 4 columns, four edges of a
// column adjacent: a cache line then holds eight edges of a slice instead of one, 32 compute units share a row of
// 128 columns, and a wave reads ahead in whole lines.  Same order, same bits.  1 M edges x 128 fp32
// columns with a row of 27 000: 428 us, now 127 and 13 for the copy.  In slices of 8 columns 142 us, and 185 without
// reading the next values from the LDS while some are summed.  Four units ahead keep the kernel at 119 registers; six
// take 129, and with them a wave per SIMD, at the same time.
constexpr int FWD_STAGED_COLS = 4;
constexpr int FWD_STAGED_UNIT = 64;         // edges per read of a slice: a kilobyte
constexpr int FWD_STAGED_ROWS = 512;        // at most
// Edges: below, the copy takes longer than it saves (262 000 edges x 128 columns, longest row of 2 190 edges: 48 us, with its
// copy 56; 2 612 edges: 56 / 50).  Rows of fewer columns have more weights beside them and are summed more slowly, 38 edges a
// microsecond with 8 heads of 8 columns (524 000 edges, rows of up to 8 400, those above 2 432 / 2 048 copied: 85 / 80 us).
constexpr int64_t FWD_STAGED_MIN = 2432, FWD_STAGED_MIN_NARROW = 2048;
constexpr int64_t FWD_STAGED_NARROW = 128;  // columns: fewer are narrow

struct FwdArgs {
  const int64_t *ptr, *idx;
  const void *vin;
  const int64_t *hmap;
  const void *hbuf;
  int hist_dtype;
  int64_t hsize;
  const uint32_t *src_bits;   // per-source substitution, nullable: one bit per source, "has an entry"
  const float *ev;
  int n_head;
  float *vout;
  int64_t R, F;
  int slots;                  // F / VEC
  bool small_matrix;          // vin holds less than 4 GiB
  int64_t split_above;        // rows with more edges are summed as four quarters (0: never)
  int64_t slice_above;        // rows with more edges belong to the front blocks, when there are any (0: none)
  SegList near, far;          // whole-row and slice-wise tasks of the front blocks
  SegList staged;             // rows that are copied side by side first, ...
  int32_t *staged_order;      // ... in their order: the rows, from FWD_STAGED_ROWS on the first unit of each copy, ...
  float *stage;               // ... and the room for that (several heads; nullable)
  int64_t stage_floats;
  int n_tiles;                // tiles of the lists; 0: every front block looks the rows through itself
  int64_t tile;
  FwdPlan *plan;              // with lists: written by the launch that makes them
  int front;                  // blocks at the start of the grid that work through the lists
};

// Rows above this many edges are shared out slice by slice; up to it a long row is one block's task.  On large
// blocks a row may take one compute unit 1/32 of the launch's time (a row of E / 8192 edges) without harm, and
// whole rows move more bytes per load.
__device__ __forceinline__ int64_t fwd_far_above(const FwdArgs &a, int64_t total) {
  const int64_t t = total / 8192;
  return a.split_above > 0 && t > a.slice_above ? t : a.slice_above;
}

// Rows above this many edges are staged: alone they would take longer (64 edges a microsecond) than the launch moves its
// rows' bytes (5 TB/s).  At most FWD_STAGED_ROWS - 1 rows are that long.
__device__ __forceinline__ int64_t fwd_staged_above(const FwdArgs &a, int64_t total) {
  int64_t t = total / 20000 * a.F;
  if (t < total / FWD_STAGED_ROWS) t = total / FWD_STAGED_ROWS;
  const int64_t least = a.F < FWD_STAGED_NARROW ? FWD_STAGED_MIN_NARROW : FWD_STAGED_MIN;
  return t < least ? least : t;
}

// The staged rows: row i's copy starts at unit unit[i] (of FWD_STAGED_UNIT edges), F + n_head floats per edge: the row's
// slices one after the other, then its weights, head by head.
struct FwdStaged {
  int32_t row[FWD_STAGED_ROWS];
  int32_t unit[FWD_STAGED_ROWS + 1];
  int32_t sum[HC_WAVES_PER_BLOCK];
};

// Exclusive sums of two values per thread over the block; `total` in every thread.
__device__ __forceinline__ void fwd_block_scan(int32_t *sum, int lane, int wave, int a0, int a1, int &x0, int &x1, int &total) {
  int incl = a0 + a1;
#pragma unroll
  for (int d = 1; d < HC_WAVE; d <<= 1) {
    const int y = __shfl_up(incl, d, HC_WAVE);
    if (lane >= d) incl += y;
  }
  __syncthreads();
  if (lane == HC_WAVE - 1) sum[wave] = incl;
  __syncthreads();
  x0 = incl - a0 - a1;
  total = 0;
#pragma unroll
  for (int w = 0; w < HC_WAVES_PER_BLOCK; ++w) {
    if (w < wave) x0 += sum[w];
    total += sum[w];
  }
  x1 = x0 + a0;
}

// Reads the list of the rows to be staged (all threads of the block).  Returns how many of them have room; they are the
// first of the list, `*n` rows, the longest first if there is not room for all: what is left takes as long as its longest
// row.  (1 M edges x 128 columns in two heads, power-law rows of up to 14 900 edges, not room for all of them: 280 us without
// copies, 208 with the first of the list and the others behind them, now 154.)  Every block of fwd_stage arrives at the
// same result; the first one writes it down for the front blocks.
__device__ __forceinline__ int fwd_read_staged(const FwdArgs &a, FwdStaged &s, int lane, int wave, int *n) {
  static_assert(SEG_MAX_REGIONS == 2 * HC_BLOCK && FWD_STAGED_ROWS == 2 * HC_BLOCK, "two tiles and two rows per thread");
  const int t = (int)threadIdx.x;
  const int c0 = 2 * t < a.n_tiles ? a.staged.count[2 * t] : 0, c1 = 2 * t + 1 < a.n_tiles ? a.staged.count[2 * t + 1] : 0;
  const int64_t listed = a.plan->listed, above = a.plan->staged_above;
  int x0, x1, rows;
  fwd_block_scan(s.sum, lane, wave, c0, c1, x0, x1, rows);
  *n = 0;
  if (listed == 0 || rows == 0) return 0;
  for (int k = 0; k < c0 + c1; ++k) {
    const int64_t part = seg_part(a.ptr, (int64_t)(k < c0 ? 2 * t : 2 * t + 1) * a.tile, above);
    s.row[x0 + k] = a.staged.item[part + (k < c0 ? k : k - c0)];
  }
  __syncthreads();
  const int64_t room = a.stage_floats / (FWD_STAGED_UNIT * (a.F + a.n_head));
  int u0, u1, all;
  const auto place = [&]() {
    const auto units = [&](int i) -> int {
      if (i >= rows) return 0;
      const int64_t r = s.row[i];
      return (int)((a.ptr[r + 1] - a.ptr[r] + FWD_STAGED_UNIT - 1) / FWD_STAGED_UNIT);
    };
    u0 = units(2 * t);
    u1 = units(2 * t + 1);
    fwd_block_scan(s.sum, lane, wave, u0, u1, x0, x1, all);
  };
  place();
  if (all > room) {
    s.unit[2 * t] = u0;
    s.unit[2 * t + 1] = u1;
    const int r0 = 2 * t < rows ? s.row[2 * t] : 0, r1 = 2 * t + 1 < rows ? s.row[2 * t + 1] : 0;
    __syncthreads();
    int p0 = 0, p1 = 0;
    for (int i = 0; i < rows; ++i) {
      const int u = s.unit[i];
      p0 += u > u0 || (u == u0 && i < 2 * t);
      p1 += u > u1 || (u == u1 && i < 2 * t + 1);
    }
    if (2 * t < rows) s.row[p0] = r0;
    if (2 * t + 1 < rows) s.row[p1] = r1;
    __syncthreads();
    place();
  }
  s.unit[2 * t] = x0;
  s.unit[2 * t + 1] = x1;
  if (t == HC_BLOCK - 1) s.unit[FWD_STAGED_ROWS] = all;
  const int fit = __syncthreads_count(2 * t < rows && x0 + u0 <= room) + __syncthreads_count(2 * t + 1 < rows && x1 + u1 <= room);
  *n = rows;
  return fit;
}

// Copies the staged rows side by side, widened to fp32: a wave takes 64 edges, 64 columns at a time, a lane one column.
template <typename T>
__global__ __launch_bounds__(HC_BLOCK) void fwd_stage(FwdArgs a) {
  __shared__ FwdStaged s;
  const int lane = hc_lane(), wave = hc_wave_in_block();
  int n;
  const int fit = fwd_read_staged(a, s, lane, wave, &n);
  if (blockIdx.x == 0) {                               // for the launch that sums
    for (int i = (int)threadIdx.x; i < n; i += HC_BLOCK) a.staged_order[i] = s.row[i];
    for (int i = (int)threadIdx.x; i <= fit && n > 0; i += HC_BLOCK) a.staged_order[FWD_STAGED_ROWS + i] = s.unit[i];
    if (threadIdx.x == 0) {
      a.plan->staged = n;
      a.plan->staged_fit = fit;
    }
  }
  if (fit == 0) return;
  const int units = s.unit[fit];
  for (int u = (int)blockIdx.x * HC_WAVES_PER_BLOCK + wave; u < units; u += (int)gridDim.x * HC_WAVES_PER_BLOCK) {
    int lo = 0, hi = fit - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s.unit[mid] <= u) lo = mid;
      else hi = mid - 1;
    }
    lo = __builtin_amdgcn_readfirstlane(lo);
    const int64_t row = s.row[lo], first = a.ptr[row];
    const int64_t e0 = (int64_t)(u - s.unit[lo]) * FWD_STAGED_UNIT, deg = a.ptr[row + 1] - first;
    const int64_t len = (int64_t)(s.unit[lo + 1] - s.unit[lo]) * FWD_STAGED_UNIT;
    float *to = a.stage + (int64_t)s.unit[lo] * FWD_STAGED_UNIT * (a.F + a.n_head);
    // behind the row's end: its last edge again, not added
    static_assert(FWD_STAGED_UNIT == HC_WAVE, "a lane per edge");
    const int64_t e = e0 + lane < deg ? e0 + lane : deg - 1;
    const int64_t at = a.idx[first + e] * a.F;
    // (lanes behind the row's last column read it again: the lanes' ids are broadcast, so all must be here)
    for (int64_t c0 = 0; c0 < a.F; c0 += HC_WAVE) {
      const int64_t c = c0 + lane < a.F ? c0 + lane : a.F - 1;
      float *col = to + c / FWD_STAGED_COLS * len * FWD_STAGED_COLS + e0 * FWD_STAGED_COLS + c % FWD_STAGED_COLS * 4;
      constexpr int AT_ONCE = 32;
      for (int i0 = 0; i0 < FWD_STAGED_UNIT; i0 += AT_ONCE) {
        T v[AT_ONCE];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) v[i] = static_cast<const T *>(a.vin)[hc_readlane64(at, i0 + i) + c];
#pragma unroll
        for (int i = 0; i < AT_ONCE; i += 4) {
          const float o[4] = {hc_to_f32<T>(v[i]), hc_to_f32<T>(v[i + 1]), hc_to_f32<T>(v[i + 2]), hc_to_f32<T>(v[i + 3])};
          if (c0 + lane < a.F) hc_store_f32<4>(col + (i0 + i) * FWD_STAGED_COLS, o);
        }
      }
    }
    float *w = to + len * a.F;
    for (int h = 0; h < a.n_head; ++h) w[h * len + e0 + lane] = a.ev[(first + e) * a.n_head + h];
  }
}

template <int N>
using FwdInt = std::integral_constant<int, N>;

template <int... I, typename F>
__device__ __forceinline__ void fwd_each(std::integer_sequence<int, I...>, F f) {
  (f(FwdInt<I>()), ...);
}

// A wave's LDS for one slice of a staged row: two units of 64 edges x 4 columns, and their weights.
struct FwdSlice {
  float x[2][FWD_STAGED_UNIT * FWD_STAGED_COLS];
  float w[2][FWD_STAGED_UNIT];
};

// Columns 4 slice .. 4 slice + 3 of staged row i, summed in edge order by one wave: every lane reads 16 bytes of a unit
// (four units ahead, into registers) and passes them through the LDS; lane l then adds up column l % 4.
__device__ __forceinline__ void fwd_sum_staged(const FwdArgs &a, FwdSlice &b, int i, int slice, int lane) {
  constexpr int AHEAD = 4;
  typedef float quad __attribute__((ext_vector_type(4)));
  const int32_t *unit = a.staged_order + FWD_STAGED_ROWS + i;
  const int64_t row = a.staged_order[i], deg = a.ptr[row + 1] - a.ptr[row];
  const int units = unit[1] - unit[0];
  const int64_t len = (int64_t)units * FWD_STAGED_UNIT;
  const float *from = a.stage + (int64_t)unit[0] * FWD_STAGED_UNIT * (a.F + a.n_head);
  const int h = (int)((int64_t)slice * FWD_STAGED_COLS / (a.F / a.n_head));
  const quad *x = reinterpret_cast<const quad *>(from + (int64_t)slice * len * FWD_STAGED_COLS) + lane;
  const float *w = from + len * a.F + h * len + lane;
  quad rx[AHEAD];
  float rw[AHEAD];
  constexpr std::make_integer_sequence<int, AHEAD> slots{};      // (a loop's counter as an index sends the arrays to scratch memory)
  const auto load = [&](auto r, int u) {
    u = u < units ? u : units - 1;
    rx[r.value] = x[(int64_t)u * HC_WAVE];
    rw[r.value] = w[(int64_t)u * FWD_STAGED_UNIT];
  };
  const auto pass = [&](auto r) {
    *reinterpret_cast<quad *>(&b.x[r.value & 1][lane * 4]) = rx[r.value];
    b.w[r.value & 1][lane] = rw[r.value];
  };
  float acc = 0.0f;
  const int c = lane & (FWD_STAGED_COLS - 1);
  // A quarter of a unit: the values of the next quarter are read from the LDS while one is summed.
  constexpr int PART = FWD_STAGED_UNIT / 4 / 4;
  quad v[2][PART], m[2][PART];
  const auto read = [&](auto r, auto part) {
#pragma unroll
    for (int q = 0; q < PART; ++q) {
      v[part.value & 1][q] = *reinterpret_cast<const quad *>(&b.x[r.value & 1][((part.value * PART + q) * FWD_STAGED_COLS + c) * 4]);
      m[part.value & 1][q] = *reinterpret_cast<const quad *>(&b.w[r.value & 1][(part.value * PART + q) * 4]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  const auto add = [&](auto part) {
#pragma unroll
    for (int q = 0; q < PART; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __fmaf_rn(v[part.value & 1][q][e], m[part.value & 1][q][e], acc);
    asm("" : "+v"(acc));      // here, not behind the next reads
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr FwdInt<0> q0;
  constexpr FwdInt<1> q1;
  constexpr FwdInt<2> q2;
  constexpr FwdInt<3> q3;
  fwd_each(slots, [&](auto r) { load(r, r.value); });
  pass(q0);
  const int whole = (int)(deg / FWD_STAGED_UNIT);
  int u = 0;
  read(q0, q0);
  for (; u + AHEAD <= whole; u += AHEAD)
    fwd_each(slots, [&](auto r) {
      constexpr FwdInt<(r.value + 1) % AHEAD> next;
      load(r, u + r.value + AHEAD);
      read(r, q1);
      add(q0);
      read(r, q2);
      add(q1);
      read(r, q3);
      add(q2);
      pass(next);
      read(next, q0);
      add(q3);
    });
  // the last units, which are on their way, and the last edges
  fwd_each(slots, [&](auto r) {
    const int64_t left = deg - (int64_t)(u + r.value) * FWD_STAGED_UNIT;
    if (left <= 0) return;
    if (r.value > 0) pass(r);
    if (left >= FWD_STAGED_UNIT) {
      read(r, q0);
      read(r, q1);
      add(q0);
      read(r, q2);
      add(q1);
      read(r, q3);
      add(q2);
      add(q3);
      return;
    }
    for (int e = 0; e < (int)left; ++e)
      acc = __fmaf_rn(b.x[r.value & 1][(e / 4 * FWD_STAGED_COLS + c) * 4 + e % 4], b.w[r.value & 1][e], acc);
  });
  if (lane < FWD_STAGED_COLS) a.vout[row * a.F + slice * FWD_STAGED_COLS + lane] = acc;
}

// Address of the neighbour row that edge `e` reads (and its weight).
// Per-source substitution: a source whose bit is clear never touches the map, which costs a whole cache line
// per lookup.  TH is the element type of the history table; when it differs from T the address carries a tag
// in its lowest bit (rows are at least 2-byte aligned) and the load of a neighbour row picks the element type
// from it -- the branch is wave-uniform, as the row address is.
template <typename T, typename TH, bool SRC>
__device__ __forceinline__ int64_t fwd_row_address(const FwdArgs &a, int64_t id) {
  int64_t addr = reinterpret_cast<int64_t>(static_cast<const T *>(a.vin) + id * a.F);
  if constexpr (SRC) {
    const bool maybe = a.src_bits == nullptr || ((a.src_bits[id >> 5] >> (id & 31)) & 1u) != 0u;
    if (maybe) {
      const int64_t slot = a.hmap[id];
      if (slot != -1)
        addr = reinterpret_cast<int64_t>(static_cast<const TH *>(a.hbuf) + slot * a.hsize) |
               (std::is_same<T, TH>::value ? 0 : 1);
    }
  }
  return addr;
}

// A neighbour row that lies in the features or, in another element type, in the history table: both are loaded, the
// one that the row does not lie in through a descriptor of no bytes, which answers with zeros and asks the memory
// nothing.  (With a branch between the two loads the compiler waits for every row before the next one's load: 14 000
// edges of a half-precision table took 0.18 us each.)
template <typename T, typename TH>
struct FwdEither {
  hc_buffer features, table;
  bool from_table;
  __device__ __forceinline__ FwdEither(int64_t address, int64_t F) {
    from_table = (address & 1) != 0;
    const void *row = reinterpret_cast<const void *>(address & ~(int64_t)1);
    features = hc_make_buffer(row, from_table ? 0u : (uint32_t)F * (uint32_t)sizeof(T));
    table = hc_make_buffer(row, from_table ? (uint32_t)F * (uint32_t)sizeof(TH) : 0u);
  }
};

// Columns of a lane: chunk k holds elements off[k] .. off[k] + VEC - 1; lanes behind the row's end read
// the last slot again (no extra line) and store nothing.
template <int VEC, int CHUNKS>
struct FwdCols {
  uint32_t off[CHUNKS];
  bool on[CHUNKS];
  int hd[CHUNKS];
  __device__ __forceinline__ FwdCols(const FwdArgs &a, int tile, int lane, bool heads) {
#pragma unroll
    for (int k = 0; k < CHUNKS; ++k) {
      const int slot = (tile * CHUNKS + k) * HC_WAVE + lane;
      on[k] = slot < a.slots;
      off[k] = (uint32_t)(on[k] ? slot : a.slots - 1) * VEC;
      hd[k] = heads ? (int)(off[k] / (uint32_t)(a.F / a.n_head)) : 0;
    }
  }
};

// Sum of the neighbour rows of edges [begin, end), added to acc in edge order by the calling wave.
// SRC (per-source substitution): neighbour rows and ids are loaded with the non-temporal hint.  Every edge
// also looks its source up in the map, and the map (not the rows, which are too many to be reused) is what
// is worth keeping in the caches.
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE>
__device__ __forceinline__ void fwd_accumulate(const FwdArgs &a, const FwdCols<VEC, CHUNKS> &col, int64_t begin,
                                               int64_t end, int lane, float (&acc)[CHUNKS][VEC]) {
  constexpr bool MIXED = SRC && !std::is_same<T, TH>::value;
  for (int64_t base = begin; base < end; base += HC_WAVE) {
    const int64_t left = end - base;
    const int n = left < HC_WAVE ? (int)left : HC_WAVE;
    // Stage: lane l resolves the address of neighbour base+l.
    int64_t my_addr = 0;
    float my_w = 0.0f;
    if (lane < n) {
      const int64_t id = SRC ? __builtin_nontemporal_load(a.idx + base + lane) : a.idx[base + lane];
      my_addr = fwd_row_address<T, TH, SRC>(a, id);
      if constexpr (WMODE == W_EDGE) my_w = a.ev[base + lane];
    }
    const auto add = [&](const auto &x, float w1, const float (&wh)[CHUNKS]) {
#pragma unroll
      for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          if constexpr (WMODE == W_NONE) acc[k][i] += x(k, i);
          else acc[k][i] = __fmaf_rn(x(k, i), WMODE == W_EDGE_HEAD ? wh[k] : w1, acc[k][i]);
        }
    };
    if constexpr (MIXED) {
      for (int j = 0; j < n; j += UNROLL) {
        float vm[UNROLL][CHUNKS][VEC];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          if (j + u < n) {
            const int64_t p = hc_readlane64(my_addr, j + u);
            if ((p & 1) != 0) {      // a row of the history table, in its own element type
              typename hc_piece<TH, VEC>::raw_t h[CHUNKS];
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k) h[k] = hc_piece<TH, VEC>::template load<true>(p - 1, col.off[k] * (uint32_t)sizeof(TH));
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
                for (int i = 0; i < VEC; ++i) vm[u][k][i] = hc_piece<TH, VEC>::widen(h[k], i);
            } else {
              typename hc_piece<T, VEC>::raw_t v[CHUNKS];
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k) v[k] = hc_piece<T, VEC>::template load<true>(p, col.off[k] * (uint32_t)sizeof(T));
#pragma unroll
              for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
                for (int i = 0; i < VEC; ++i) vm[u][k][i] = hc_piece<T, VEC>::widen(v[k], i);
            }
          }
        }
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
          if (j + u < n) add([&](int k, int i) { return vm[u][k][i]; }, 0.0f, {});
      }
    } else {
      typename hc_piece<T, VEC>::raw_t v[UNROLL][CHUNKS];
      float wh[WMODE == W_EDGE_HEAD ? UNROLL : 1][CHUNKS];
      // COUNT rows from place `at` of the stage into slots SLOT ... ; loads first, then the adds in order
      const auto load = [&](auto slot, auto count, int at) {
#pragma unroll
        for (int k = 0; k < CHUNKS; ++k) {
          uint32_t byte = col.off[k] * (uint32_t)sizeof(T);
          asm("" : "+v"(byte));      // seen as 32 bits beside the loads, which then take the row's address from scalar registers
#pragma unroll
          for (int u = 0; u < count.value; ++u)
            v[slot.value + u][k] = hc_piece<T, VEC>::template load<SRC>(hc_readlane64(my_addr, at + u), byte);
        }
        if constexpr (WMODE == W_EDGE_HEAD) {
#pragma unroll
          for (int u = 0; u < count.value; ++u)
#pragma unroll
            for (int k = 0; k < CHUNKS; ++k) wh[slot.value + u][k] = a.ev[(base + at + u) * a.n_head + col.hd[k]];
        }
      };
      const auto sum = [&](auto slot, auto count, int at) {
#pragma unroll
        for (int u = 0; u < count.value; ++u) {
          const float w1 = WMODE == W_EDGE ? hc_readlane_f(my_w, at + u) : 0.0f;
          add([&](int k, int i) { return hc_piece<T, VEC>::widen(v[slot.value + u][k], i); }, w1,
              wh[WMODE == W_EDGE_HEAD ? slot.value + u : 0]);
        }
      };
      int j = 0;
      for (; j + UNROLL <= n; j += UNROLL) {
        load(FwdInt<0>(), FwdInt<UNROLL>(), j);
        sum(FwdInt<0>(), FwdInt<UNROLL>(), j);
      }
      // the rest in parts of 8, 4, 2 and 1, all of their loads first.  (Asking of every row of a batch whether it is
      // there took five scalar instructions a row: 1 M rows of 3 edges of 64 columns 443 us instead of 336.)
      const int rest = n - j;
      if (rest > 0) {
        const int j4 = j + (rest & 8), j2 = j4 + (rest & 4), j1 = j2 + (rest & 2);
        constexpr FwdInt<0> s8;
        constexpr FwdInt<UNROLL - 8> s4;      // slots behind the larger parts'
        constexpr FwdInt<UNROLL - 4> s2;
        constexpr FwdInt<UNROLL - 2> s1;
        if constexpr (UNROLL > 8)
          if ((rest & 8) != 0) load(s8, FwdInt<8>(), j);
        if constexpr (UNROLL > 4)
          if ((rest & 4) != 0) load(s4, FwdInt<4>(), j4);
        if ((rest & 2) != 0) load(s2, FwdInt<2>(), j2);
        if ((rest & 1) != 0) load(s1, FwdInt<1>(), j1);
        if constexpr (UNROLL > 8)
          if ((rest & 8) != 0) sum(s8, FwdInt<8>(), j);
        if constexpr (UNROLL > 4)
          if ((rest & 4) != 0) sum(s4, FwdInt<4>(), j4);
        if ((rest & 2) != 0) sum(s2, FwdInt<2>(), j2);
        if ((rest & 1) != 0) sum(s1, FwdInt<1>(), j1);
      }
    }
  }
}

// SV adjacent columns per lane of edges [begin, end), summed in edge order with D to 2 D rows in flight: the loads of
// a group of D rows are issued before the adds of the group in front of it, and the ids of the next 64 edges
// before the rows of these.  (Straight-line code over whole stages of 64 edges: only then can a wave wait for
// the older group alone.  A wave on its own is bound by the latency of its groups: 20 000 edges of 64 fp32
// columns took 390 us with eight rows in flight and one wait for all of them.)
// W_EDGE: the weight of edge e is ev[e * ev_stride] (rows of several heads whose slice lies in one head).
// BUF: the matrix is smaller than 4 GiB and its rows are addressed by 32-bit offsets (a wave on its own issues
// one instruction in four cycles: with 64-bit row addresses the eleven instructions per edge took 23 ns).
template <typename T, typename TH, int SV, bool SRC, int WMODE, int D, bool BUF>
__device__ __forceinline__ void fwd_slice_sum(const FwdArgs &a, uint32_t c, int64_t begin, int64_t end, int lane,
                                              const float *__restrict__ ev, int64_t ev_stride, float (&acc)[SV]) {
  static_assert(!BUF || !SRC, "the substituted rows lie in another matrix");
  constexpr int G = HC_WAVE / D;
  constexpr bool MIXED = SRC && !std::is_same<T, TH>::value;
  typedef typename hc_piece<T, SV>::raw_t raw_t;
  const int hd = WMODE == W_EDGE_HEAD ? (int)(c / (uint32_t)(a.F / a.n_head)) : 0;
#pragma unroll
  for (int i = 0; i < SV; ++i) acc[i] = 0.0f;
  if (begin >= end) return;
  const hc_buffer buf = hc_make_buffer(a.vin);
  const uint32_t row_bytes = (uint32_t)a.F * (uint32_t)sizeof(T);
  const auto address = [&](int64_t id) -> int64_t {
    if constexpr (BUF) return (int64_t)((uint32_t)id * row_bytes);
    else return fwd_row_address<T, TH, SRC>(a, id);
  };
  // MIXED: the table's share of a row (see FwdEither), and the stage's edges that read the table
  uint16_t yb[2][MIXED ? D : 1];
  unsigned long long tables = 0ull, next_tables = 0ull;
  const auto load = [&](raw_t (&x)[D], float (&w)[D], uint16_t (&y)[MIXED ? D : 1], int64_t addr, int64_t base, int g,
                        int last) {
    uint32_t off[D];
    if constexpr (BUF) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        const int j = g * D + u;
        off[u] = (uint32_t)__builtin_amdgcn_readlane((int)addr, j < last ? j : last);
      }
    }
#pragma unroll
    for (int u = 0; u < D; ++u) {
      int j = g * D + u;
      j = j < last ? j : last;                                 // behind the end: the last row again, not added
      if constexpr (BUF) {
        x[u] = hc_buffer_load<raw_t>(buf, c * (uint32_t)sizeof(T), off[u]);
      } else {
        const int64_t p = hc_readlane64(addr, j);
        if constexpr (MIXED) {
          static_assert(!MIXED || SV == 1, "a table of another element type beside fp32 rows");
          const FwdEither<T, TH> row(p, a.F);
          x[u] = hc_buffer_load_nt<raw_t>(row.features, c * (uint32_t)sizeof(T));
          y[u] = hc_buffer_load_nt<uint16_t>(row.table, c * (uint32_t)sizeof(TH));
        } else {
          x[u] = hc_piece<T, SV>::template load<SRC>(p, c * (uint32_t)sizeof(T));
        }
      }
      if constexpr (WMODE == W_EDGE_HEAD) w[u] = ev[(base + j) * a.n_head + hd];
    }
  };
  const auto add1 = [&](const raw_t &x, float w, uint16_t y, float my_w, int j) {
    const float w1 = WMODE == W_EDGE ? hc_readlane_f(my_w, j) : w;
#pragma unroll
    for (int i = 0; i < SV; ++i) {
      if constexpr (MIXED)
        acc[i] += ((tables >> j) & 1ull) != 0ull ? hc_piece<TH, 1>::widen(y, 0) : hc_piece<T, SV>::widen(x, i);
      else if constexpr (WMODE == W_NONE) acc[i] += hc_piece<T, SV>::widen(x, i);
      else acc[i] = __fmaf_rn(hc_piece<T, SV>::widen(x, i), w1, acc[i]);
    }
  };
  raw_t x[2][D];
  float w[2][D];
  int64_t e = begin + lane < end ? begin + lane : end - 1;
  int64_t addr = address(a.idx[e]);
  if constexpr (MIXED) tables = __ballot((addr & 1) != 0);
  float my_w = WMODE == W_EDGE ? ev[e * ev_stride] : 0.0f;
  int last = end - begin < HC_WAVE ? (int)(end - begin) - 1 : HC_WAVE - 1;
  load(x[0], w[0], yb[0], addr, begin, 0, last);
  int64_t base = begin;
  for (; base + HC_WAVE <= end; base += HC_WAVE) {
    const int64_t next = base + HC_WAVE;
    e = next + lane < end ? next + lane : end - 1;
    const int64_t next_id = a.idx[e];
    const float next_w = WMODE == W_EDGE ? ev[e * ev_stride] : 0.0f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G) {
        load(x[(g + 1) & 1], w[(g + 1) & 1], yb[(g + 1) & 1], addr, base, g + 1, HC_WAVE - 1);
      } else {
        addr = address(next_id);
        if constexpr (MIXED) next_tables = __ballot((addr & 1) != 0);
        last = end - next < HC_WAVE ? (int)(end - next) - 1 : HC_WAVE - 1;
        last = last < 0 ? 0 : last;
        load(x[0], w[0], yb[0], addr, next < end ? next : end - 1, 0, last);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < D; ++u) add1(x[g & 1][u], w[g & 1][u], yb[g & 1][MIXED ? u : 0], my_w, g * D + u);
      __builtin_amdgcn_sched_barrier(0);
    }
    my_w = next_w;
    if constexpr (MIXED) tables = next_tables;
  }
  // the last, partial stage: its first group is on its way
  const int n = (int)(end - base);
  for (int g = 0; g * D < n; ++g) {
    if (g > 0) load(x[0], w[0], yb[0], addr, base, g, n - 1);
#pragma unroll
    for (int u = 0; u < D; ++u)
      if (g * D + u < n) add1(x[0][u], w[0][u], yb[0][MIXED ? u : 0], my_w, g * D + u);
  }
}

template <typename T, typename TH, int SV, bool SRC, int WMODE, int D>
__device__ __forceinline__ void fwd_slice_any(const FwdArgs &a, uint32_t c, int64_t begin, int64_t end, int lane,
                                              const float *__restrict__ ev, int64_t ev_stride, float (&acc)[SV]) {
  if constexpr (!SRC) {
    if (a.small_matrix) {
      fwd_slice_sum<T, TH, SV, SRC, WMODE, D, true>(a, c, begin, end, lane, ev, ev_stride, acc);
      return;
    }
  }
  fwd_slice_sum<T, TH, SV, SRC, WMODE, D, false>(a, c, begin, end, lane, ev, ev_stride, acc);
}

// A block owns four consecutive destination rows, one per wave.  Rows of up to 256 edges are summed by
// their wave, in CSR order.  Longer rows are split into four contiguous quarters (quarter length
// ceil(deg/4)), each summed in CSR order, and combined left to right, ((q0 + q1) + q2) + q3, before the
// division: by the front blocks of the grid when the rows were listed (see seg_list.h), else by the four
// waves of the row's own block behind its other rows.
constexpr int FWD_ROWS_PER_BLOCK = HC_WAVES_PER_BLOCK;
constexpr int FWD_XCD_CHUNK = 256;  // consecutive blocks (1024 rows) that share an XCD

// One long row summed by the four waves of the calling block (all of them must call this), whole rows per
// load: wave w takes the w-th quarter.
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE>
__device__ __forceinline__ void fwd_long_row(const FwdArgs &a, int64_t lrow, int lane, int wave,
                                             float (*part)[HC_WAVE * VEC * CHUNKS]) {
  const int64_t lb = a.ptr[lrow];
  const int64_t le = a.ptr[lrow + 1];
  const int64_t deg = le - lb;
  const int64_t q = (deg + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
  int64_t sb = lb + wave * q;
  int64_t se = sb + q;
  if (sb > le) sb = le;
  if (se > le) se = le;
  const int tiles = (a.slots + HC_WAVE * CHUNKS - 1) / (HC_WAVE * CHUNKS);
  for (int tile = 0; tile < (CHUNKS == 4 ? tiles : 1); ++tile) {
    const FwdCols<VEC, CHUNKS> col(a, tile, lane, false);
    float acc[CHUNKS][VEC];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[c][i] = 0.0f;
    fwd_accumulate<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE>(a, col, sb, se, lane, acc);
    if (wave > 0) {
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
        for (int i = 0; i < VEC; ++i) part[wave - 1][(c * HC_WAVE + lane) * VEC + i] = acc[c][i];
    }
    __syncthreads();
    if (wave == 0) {
      const float fdeg = (float)(int)deg;
      float *__restrict__ orow = a.vout + lrow * a.F;
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) {
        float o[VEC];
#pragma unroll
        for (int i = 0; i < VEC; ++i) {
          float t2 = acc[c][i];
#pragma unroll
          for (int pw = 0; pw < HC_WAVES_PER_BLOCK - 1; ++pw) t2 += part[pw][(c * HC_WAVE + lane) * VEC + i];
          o[i] = WMODE != W_NONE ? t2 : (deg > 0 ? t2 / fdeg : 0.0f);
        }
        if (col.on[c]) {
          if constexpr (SRC) hc_store_f32_nt<VEC>(orow + col.off[c], o);
          else hc_store_f32<VEC>(orow + col.off[c], o);
        }
      }
    }
    __syncthreads();
  }
}

// A slice is one cache line of a row: 32 fp32 columns, or 64 of a half-precision row in 32 lanes of two (a
// wave-wide load of single half-precision elements takes the address unit three times as long as one of whole
// words: 350 us instead of 150 us for 20 000 edges).  Half-precision rows of odd length, whose elements cannot be
// paired, are loaded one by one.
constexpr int FWD_SLICE_LANES = 32;

// Blocks of at most this many rows need no lists: their front blocks look the rows through themselves.
constexpr int64_t FWD_SELF_ROWS = 4096;
constexpr int FWD_SELF_ITEMS = 512;

// The front blocks: slices of the longest rows (one block per task, wave = quarter; rows of several heads: one
// wave per task), then the other listed rows as whole rows.
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE>
__device__ __forceinline__ void fwd_front(const FwdArgs &a, int64_t far_above, int lane, int wave,
                                          float (*part)[HC_WAVE * VEC * CHUNKS], int *self_rows, int *self_n,
                                          FwdSlice *slice) {
  constexpr int SV = sizeof(T) == 2 && VEC > 1 ? 2 : 1;
  constexpr int SL = FWD_SLICE_LANES * SV;
  const int ns = (int)((a.F + SL - 1) / SL);
  SegIndex far_index;
  int n_far;
  if (a.n_tiles > 0) {
    far_index = seg_index(a.far.count, a.n_tiles, lane);
    n_far = far_index.total;
  } else {
    // Few rows: look them through here (at most FWD_SELF_ITEMS of them can be long, see `listed`).  Wave w takes
    // a contiguous run of rows and the runs are joined in order, so that every block arrives at the same list.
    constexpr int IT = (int)(FWD_SELF_ROWS / HC_BLOCK);
    unsigned long long m[IT];
    int mine = 0;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int64_t r = ((int64_t)wave * IT + it) * HC_WAVE + lane;
      const bool is_long = r < a.R && a.ptr[r + 1] - a.ptr[r] > far_above && (SRC || a.hmap == nullptr || a.hmap[r] == -1);
      m[it] = __ballot(is_long);
      mine += __popcll(m[it]);
    }
    if (lane == 0) self_n[wave] = mine;
    __syncthreads();
    int at = 0;
    n_far = 0;
#pragma unroll
    for (int w = 0; w < HC_WAVES_PER_BLOCK; ++w) {
      if (w < wave) at += self_n[w];
      n_far += self_n[w];
    }
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      if ((m[it] >> lane) & 1ull) self_rows[at + __popcll(m[it] & below)] = (wave * IT + it) * HC_WAVE + lane;
      at += __popcll(m[it]);
    }
    __syncthreads();
  }
  const auto far_row = [&](int e) -> int64_t {
    if (a.n_tiles == 0) return (int64_t)__builtin_amdgcn_readfirstlane(self_rows[e]);
    int t, w;
    seg_locate(far_index, e, &t, &w);
    return (int64_t)__builtin_amdgcn_readfirstlane(a.far.item[seg_part(a.ptr, (int64_t)t * a.tile, far_above) + w]);
  };
  // the lane's columns of slice `sl`; lanes behind the slice or the row read its last ones again
  const auto columns = [&](int sl, bool &on) -> uint32_t {
    const int c = (sl * FWD_SLICE_LANES + (lane < FWD_SLICE_LANES ? lane : FWD_SLICE_LANES - 1)) * SV;
    on = lane < FWD_SLICE_LANES && c < a.F;
    return (uint32_t)(c < a.F ? c : a.F - SV);
  };
  const int64_t tasks = (int64_t)n_far * ns;
  if constexpr (WMODE == W_EDGE_HEAD) {                  // rows of several heads are never split: one wave per task
    const auto slice_of = [&](int64_t row, int sl) {
      bool on;
      const uint32_t c = columns(sl, on);
      const int64_t b = a.ptr[row], e = a.ptr[row + 1];
      float s[SV];
      // every column of the slice in one head: its weights are staged with the ids, 64 at a time
      const int fh = (int)(a.F / a.n_head);
      const int c0 = sl * SL;
      const int c1 = (c0 + SL < a.F ? c0 + SL : (int)a.F) - 1;
      if (c0 / fh == c1 / fh)
        fwd_slice_any<T, TH, SV, SRC, W_EDGE, 32>(a, c, b, e, lane, a.ev + c0 / fh, a.n_head, s);
      else
        fwd_slice_sum<T, TH, SV, SRC, W_EDGE_HEAD, 16, false>(a, c, b, e, lane, a.ev, 0, s);
#pragma unroll
      for (int i = 0; i < SV; ++i)
        if (on) a.vout[row * a.F + c + i] = s[i];
    };
    // wave 0 of every block has the copied rows; those without room begin with wave 1 then, the other listed ones with wave 2
    int turn = wave;
    if (a.stage != nullptr && a.plan->staged > 0) {
      const int rows = (int)a.plan->staged, fit = (int)a.plan->staged_fit;
      const int pieces = (int)(a.F / FWD_STAGED_COLS);
      if (wave == 0)
        for (int64_t t = blockIdx.x; t < (int64_t)fit * pieces; t += a.front)
          fwd_sum_staged(a, *slice, (int)(t / pieces), (int)(t % pieces), lane);
      const int next = (wave + 3) % HC_WAVES_PER_BLOCK;
      for (int64_t t = (int64_t)next * a.front + blockIdx.x; t < (int64_t)(rows - fit) * ns; t += (int64_t)HC_WAVES_PER_BLOCK * a.front)
        slice_of((int64_t)a.staged_order[fit + (int)(t / ns)], (int)(t % ns));
      if (fit > 0) turn = (wave + 2) % HC_WAVES_PER_BLOCK;
    }
    for (int64_t t = (int64_t)turn * a.front + blockIdx.x; t < tasks; t += (int64_t)HC_WAVES_PER_BLOCK * a.front)
      slice_of(far_row((int)(t / ns)), (int)(t % ns));
    return;
  } else {
    for (int64_t t = blockIdx.x; t < tasks; t += a.front) {
      const int64_t row = far_row((int)(t / ns));
      bool on;
      const uint32_t c = columns((int)(t % ns), on);
      const int64_t lb = a.ptr[row], le = a.ptr[row + 1];
      const int64_t q = (le - lb + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
      int64_t sb = lb + wave * q, se = sb + q;
      if (sb > le) sb = le;
      if (se > le) se = le;
      float s[SV];
      fwd_slice_any<T, TH, SV, SRC, WMODE, 16>(a, c, sb, se, lane, a.ev, 1, s);
      if (wave > 0 && lane < FWD_SLICE_LANES) {
#pragma unroll
        for (int i = 0; i < SV; ++i) part[wave - 1][lane * SV + i] = s[i];
      }
      __syncthreads();
      if (wave == 0 && on) {
#pragma unroll
        for (int i = 0; i < SV; ++i) {
#pragma unroll
          for (int pw = 0; pw < HC_WAVES_PER_BLOCK - 1; ++pw) s[i] += part[pw][lane * SV + i];
          a.vout[row * a.F + c + i] = WMODE != W_NONE ? s[i] : s[i] / (float)(int)(le - lb);
        }
      }
      __syncthreads();
    }
    if (a.n_tiles == 0) return;
    const SegIndex near_index = seg_index(a.near.count, a.n_tiles, lane);
    for (int t = (int)blockIdx.x; t < near_index.total; t += a.front) {
      int tile, w;
      seg_locate(near_index, t, &tile, &w);
      const int64_t row = (int64_t)__builtin_amdgcn_readfirstlane(
          a.near.item[seg_part(a.ptr, (int64_t)tile * a.tile, a.slice_above) + w]);
      fwd_long_row<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE>(a, row, lane, wave, part);
    }
  }
}

// PART: the front blocks and the rows' in one launch, or one of the two.  A table of another element type beside the
// features takes two launches: the slices' code needs 170 registers there, which would leave the rows three waves per
// SIMD (11 M edges x 128 in one launch 2.55 ms, in two 1.96 ms).
constexpr int FWD_ALL = 0, FWD_FRONT = 1, FWD_BODY = 2;
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE, int PART>
__device__ __forceinline__ void fwd_block(const FwdArgs &a) {
  // without heads the rows may be split: the split code is compiled for those modes only
  constexpr int LMODE = WMODE == W_EDGE_HEAD ? W_EDGE : WMODE;
  __shared__ float part[HC_WAVES_PER_BLOCK - 1][HC_WAVE * VEC * CHUNKS];
  __shared__ int self_rows[FWD_SELF_ITEMS];
  __shared__ int long_rows[FWD_ROWS_PER_BLOCK];    // (front blocks: the waves' counts)
  FwdSlice *slice = nullptr;
  if constexpr (WMODE == W_EDGE_HEAD) {
    __shared__ __attribute__((aligned(16))) FwdSlice slice_s;
    slice = &slice_s;
  }
  __shared__ int n_long_s;
  const int lane = hc_lane();
  const int wave = hc_wave_in_block();
  // every thread of the grid reads the same words, so the decision is uniform: the lists hold every long row
  int64_t far_above = 0;
  bool listed = false;
  if (a.front > 0) {
    if (a.n_tiles > 0) {
      far_above = a.plan->far_above;
      listed = a.plan->listed != 0;
    } else {
      const int64_t total = a.ptr[a.R] - a.ptr[0];
      far_above = fwd_far_above(a, total);
      listed = total < (FWD_SELF_ITEMS + 1) * (far_above + 1) && far_above == a.slice_above;
    }
    if constexpr (PART != FWD_BODY) {
      if ((int)blockIdx.x < a.front) {
        if (listed)
          fwd_front<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE>(a, far_above, lane, wave, part, self_rows, long_rows, slice);
        return;
      }
    }
  }
  if constexpr (PART == FWD_FRONT) return;
  const int ahead = PART == FWD_BODY ? 0 : a.front;
  const int64_t row0 = hc_xcd_block<FWD_XCD_CHUNK>((int64_t)blockIdx.x - ahead, (int64_t)gridDim.x - ahead) *
                       FWD_ROWS_PER_BLOCK;
  const int64_t rest = a.R - row0;
  const int nrows = rest < FWD_ROWS_PER_BLOCK ? (int)rest : FWD_ROWS_PER_BLOCK;
  const bool in_block = a.split_above > 0 && !listed;      // the block sums its own long rows afterwards

  if (in_block) {
    if (threadIdx.x == 0) n_long_s = 0;
    __syncthreads();
  }

  if (wave < nrows) {
    const int64_t row = row0 + wave;
    float *__restrict__ orow = a.vout + row * a.F;
    bool hist = false;
    if (!SRC && a.hmap != nullptr) hist = a.hmap[row] != -1;
    if (hist) {
      if (WMODE == W_EDGE_HEAD && a.hsize != a.F) {      // one history row shared by the heads
        const int64_t fh = a.F / a.n_head;
        for (int h = 0; h < a.n_head; ++h) copy_row_any(a.hbuf, a.hist_dtype, row * a.hsize, orow + h * fh, fh, lane);
      } else {
        copy_row_any(a.hbuf, a.hist_dtype, row * a.hsize, orow, a.F, lane);
      }
    } else {
      const int64_t begin = a.ptr[row];
      const int64_t end = a.ptr[row + 1];
      const int64_t deg = end - begin;
      if (listed && deg > a.slice_above) {
        // summed by the front blocks
      } else if (in_block && deg > a.split_above) {
        if (lane == 0) long_rows[atomicAdd(&n_long_s, 1)] = wave;
      } else {
        const int tiles = (a.slots + HC_WAVE * CHUNKS - 1) / (HC_WAVE * CHUNKS);
        for (int tile = 0; tile < (CHUNKS == 4 ? tiles : 1); ++tile) {
          const FwdCols<VEC, CHUNKS> col(a, tile, lane, WMODE == W_EDGE_HEAD);
          float acc[CHUNKS][VEC];
#pragma unroll
          for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[c][i] = 0.0f;
          fwd_accumulate<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE>(a, col, begin, end, lane, acc);
          const float fdeg = (float)(int)deg;
#pragma unroll
          for (int c = 0; c < CHUNKS; ++c) {
            float o[VEC];
#pragma unroll
            for (int i = 0; i < VEC; ++i) o[i] = WMODE != W_NONE ? acc[c][i] : (deg > 0 ? acc[c][i] / fdeg : 0.0f);
            if (col.on[c]) {
              if constexpr (SRC) hc_store_f32_nt<VEC>(orow + col.off[c], o);
              else hc_store_f32<VEC>(orow + col.off[c], o);
            }
          }
        }
      }
    }
  }
  if (!in_block) return;  // the whole grid takes the same branch
  __syncthreads();
  const int n_long = n_long_s;
  // The order in which long rows were noted does not matter: each is summed on its own.
  for (int t = 0; t < n_long; ++t)
    fwd_long_row<T, TH, VEC, CHUNKS, UNROLL, SRC, LMODE>(a, row0 + long_rows[t], lane, wave, part);
}

// Plain rows, and rows beside a table of another element type: at most 80 scalar registers;
// above, fewer waves fit the chip.  (The slices would take 106, and with them 1 M rows of 3 edges of 64 columns 433 us
// instead of 388, 700 k rows of 20 edges 664 instead of 638; 6 M edges x 100 beside a half-precision table 1214 us
// instead of 1063.)
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE, int PART>
__global__ __launch_bounds__(HC_BLOCK) __attribute__((amdgpu_num_sgpr(80))) void fwd_rows(FwdArgs a) {
  fwd_block<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE, PART>(a);
}

// Weights, substituted sources: with the heads' and the substitution's vector registers there is room for four or five
// waves whatever the scalar ones, and the slices are the faster with more of these (20 M edges x 256 over 20 GB 4.19 ms,
// 4.24 with 80; a row of 27 000 weighted edges x 256 198 us, 202 with 80).
template <typename T, typename TH, int VEC, int CHUNKS, int UNROLL, bool SRC, int WMODE, int PART>
__global__ __launch_bounds__(HC_BLOCK) void fwd_rows_wide(FwdArgs a) {
  fwd_block<T, TH, VEC, CHUNKS, UNROLL, SRC, WMODE, PART>(a);
}

// One translation unit each (the kernels take a minute to compile).
__attribute__((visibility("hidden"))) int fwd_dispatch_f32(FwdArgs &a, bool src_mode, int n_head, hipStream_t st);
__attribute__((visibility("hidden"))) int fwd_dispatch_f16(FwdArgs &a, bool src_mode, int n_head, hipStream_t st);
__attribute__((visibility("hidden"))) int fwd_dispatch_bf16(FwdArgs &a, bool src_mode, int n_head, hipStream_t st);

#ifdef FWD_INSTANTIATE
namespace {

constexpr int FWD_STAGE_BLOCKS = 512;

template <typename T, int VEC, int CHUNKS>
int launch_rows(const FwdArgs &a, bool src_mode, hipStream_t st) {
  constexpr int per = VEC * CHUNKS;
  constexpr int UNROLL = per >= 16 ? 4 : (per >= 4 ? 8 : 16);
  const int64_t row_blocks = (a.R + FWD_ROWS_PER_BLOCK - 1) / FWD_ROWS_PER_BLOCK;
  const int64_t blocks = row_blocks + a.front;
  if (!hc_grid_ok(blocks)) return HC_EUNSUPPORTED;
  const dim3 grid((unsigned)blocks), block(HC_BLOCK);
#define HC_FWD_LAUNCH(WMODE) fwd_rows<T, T, VEC, CHUNKS, UNROLL, false, WMODE, FWD_ALL><<<grid, block, 0, st>>>(a)
#define HC_FWD_LAUNCH_WIDE(SRC, WMODE) fwd_rows_wide<T, T, VEC, CHUNKS, UNROLL, SRC, WMODE, FWD_ALL><<<grid, block, 0, st>>>(a)
#define HC_FWD_LAUNCH_TWO(TH)                                                                                           \
  {                                                                                                                     \
    if (a.front > 0)                                                                                                    \
      fwd_rows<T, TH, VEC, CHUNKS, UNROLL, true, W_NONE, FWD_FRONT><<<dim3((unsigned)a.front), block, 0, st>>>(a);      \
    fwd_rows<T, TH, VEC, CHUNKS, UNROLL, true, W_NONE, FWD_BODY><<<dim3((unsigned)row_blocks), block, 0, st>>>(a);      \
  }
  if (a.ev != nullptr && a.n_head > 1) {
    if (a.stage != nullptr) fwd_stage<T><<<dim3(FWD_STAGE_BLOCKS), block, 0, st>>>(a);
    HC_FWD_LAUNCH_WIDE(false, W_EDGE_HEAD);
  }
  else if (a.ev != nullptr) HC_FWD_LAUNCH_WIDE(false, W_EDGE);
  else if (src_mode && a.hmap != nullptr) {
    // the table of a per-source substitution may be narrower than fp32 features
    if constexpr (std::is_same<T, float>::value) {
      if (a.hist_dtype == HC_F16) HC_FWD_LAUNCH_TWO(__half)
      else if (a.hist_dtype == HC_BF16) HC_FWD_LAUNCH_TWO(__hip_bfloat16)
      else HC_FWD_LAUNCH_WIDE(true, W_NONE);
    } else HC_FWD_LAUNCH_WIDE(true, W_NONE);
  } else HC_FWD_LAUNCH(W_NONE);
#undef HC_FWD_LAUNCH
#undef HC_FWD_LAUNCH_WIDE
#undef HC_FWD_LAUNCH_TWO
  return hc_launch_status();
}

template <typename T, int VEC>
int launch_chunks(const FwdArgs &a, bool src_mode, hipStream_t st) {
  const int chunks = (a.slots + HC_WAVE - 1) / HC_WAVE;
  if (chunks <= 1) return launch_rows<T, VEC, 1>(a, src_mode, st);
  if (chunks == 2) return launch_rows<T, VEC, 2>(a, src_mode, st);
  if (chunks == 3) return launch_rows<T, VEC, 3>(a, src_mode, st);
  return launch_rows<T, VEC, 4>(a, src_mode, st);       // wider rows: column tiles of 256 slots
}

// Elements per lane and load: the widest power of two that the row length, a head's width and the pointers
// allow, halved while the row still fits the wave (all lanes busy rather than wide loads by a few) and a lane
// loads at least a word (loads of single half-precision elements are slow, see FWD_SLICE_LANES).
template <typename T>
int dispatch(FwdArgs &a, bool src_mode, int n_head, hipStream_t st) {
  const int64_t fh = a.F / n_head;
  const size_t hesz = a.hist_dtype == HC_F32 ? 4 : 2;
  const auto fits = [&](int v) {
    if (fh % v != 0) return false;
    if (reinterpret_cast<uintptr_t>(a.vin) % (v * sizeof(T)) != 0) return false;
    if (reinterpret_cast<uintptr_t>(a.vout) % (v > 4 ? 16 : v * sizeof(float)) != 0) return false;
    if (src_mode && a.hmap != nullptr &&
        (reinterpret_cast<uintptr_t>(a.hbuf) % (v * hesz) != 0 || a.hsize % v != 0)) return false;
    return true;
  };
  int v = 16 / (int)sizeof(T);
  while (v > 1 && (!fits(v) || (a.F / (v / 2) <= HC_WAVE && v * sizeof(T) > 4))) v /= 2;
  if (a.F / v > 0x3fffffffLL) return HC_EUNSUPPORTED;
  a.slots = (int)(a.F / v);
  if constexpr (sizeof(T) == 2)
    if (v == 8) return launch_chunks<T, 8>(a, src_mode, st);
  if (v == 4) return launch_chunks<T, 4>(a, src_mode, st);
  if (v == 2) return launch_chunks<T, 2>(a, src_mode, st);
  return launch_chunks<T, 1>(a, src_mode, st);
}

}  // namespace
#endif  // FWD_INSTANTIATE
