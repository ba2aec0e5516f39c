// Weight gradient of a layer's linear maps: dW[H, F] = g^T x for g [n, H], x [n, F] (fp32), n = rows of a
// sampled layer (thousands to a hundred thousand), H and F a few hundred.  What torch's autograd computes
// for `self.lin_l(out)` and `self.lin_r(x[:num_node])` (/root/reference/hiscache/history_model.py:94-98)
// as one GEMM each.  A short, wide product with a very long inner dimension: the work is split over the
// rows, every block multiplies its slab of rows on the matrix cores into a partial tile, and a second launch
// adds the slabs' tiles in slab order.  Two operands that share g (the aggregated rows and the root rows) go
// through the same launches.  No atomics: the result does not depend on scheduling.
//
// hc_linear_grad also takes any number of outputs (columns behind H are zeros) and adds up the columns of g, the bias' gradient,
// from the tiles that it stages anyway: a last layer of 1 000 rows, 172 classes, 256 inputs took two library GEMMs and a
// matrix-vector product, 31 us, and takes the same two launches, 13 us.
// Bound by the matrix pipes (see dense.hip) where the rows are many, by the partial tiles' way through memory and two
// launches where they are few.  Both launches, two operands, each wave loading its rows straight into registers (the
// form before: tiles of 256 x 64, one block per compute unit) / this: 1 000 rows, 256 x 128 12.6 / 9.1 us; 3 000, 256 x 256
// 24.7 / 20.9; 25 800, 256 x 128 44.6 / 40.8; 200 000, 256 x 128 272 / 248 (106 TFLOP/s); 89 000, 64 x 64 65 / 30 (three of
// its four waves had no work); one operand, 4 200 rows, 3 840 x 256 138 / 88.  Tiles of 128 x 64 and 128 x 128, pieces of
// 16 rows, 512 or 2 048 blocks instead of 1 024: between 5% faster and 40% slower, and 512 blocks sum twice the rows in one
// chain.  Slabs of 64 rows at least: with 128, 1 500 rows of 256 x 256 take 14 instead of 16 us but a tenth more error.
//
// A block of four waves stages pieces of WG_PIECE rows of g and of x through two LDS buffers, the loads of a piece
// issued in front of the matrix instructions of the one before it and kept there by a scheduling barrier.  Both
// operands lie in LDS as in memory, the row index outside; a staged row is 16 words longer than the tile, so that the
// 4 rows x 16 columns that a wave reads at once lie in 64 banks.  Rows behind the slab are read through a buffer
// descriptor that ends there and are zeros.
//
//   A operand (16 x 4): x[row k + l / 16][f0 + l % 16]        B operand (4 x 16): g[row k + l / 16][h0 + l % 16]
//   D (16 x 16, 4 values per lane): dW row h0 + l % 16, columns f0 + 4 (l / 16) .. + 3: one 16-byte store
#include "hc_common.h"

namespace {

typedef float wg_acc __attribute__((ext_vector_type(4)));
typedef uint32_t wg_quad __attribute__((ext_vector_type(4)));

constexpr int WG_TILE_H = 64;       // rows of dW per block
constexpr int WG_TILE_F = 64;       // columns of dW per block
constexpr int WG_PIECE = 32;        // rows of g and x per piece
constexpr int WG_TARGET_BLOCKS = 1024;
constexpr int WG_MIN_SLAB_ROWS = 64;
// Rows summed in one chain; a slab's chains are added one after the other, so that the error does not grow with the slab
// (a wide dW has few slabs: 30 000 rows, 3 840 x 256 are five of 6 000).  Error against 64 bits, one chain per slab / chains of
// 1 024, 512, 256 rows: 30 000 rows, 1 280 x 256 8.6e-7 / 5.5, 4.0, 3.0e-7; 200 000, 256 x 256, two operands 14.1e-7 / 5.7, 4.1,
// 3.1e-7 (batched library products over 1 024 rows each: 5.8e-7); the time is the same (200 000, 256 x 256 515 / 526 us).
constexpr int WG_CHAIN_ROWS = 256;

struct WgShape {
  int tiles_h, tiles_f;
  int64_t slab_rows, slabs;
};

static bool wg_shape(int64_t n, int64_t H, int64_t F, int n_op, WgShape *s) {
  if (n < 1 || H < 1 || F < WG_TILE_F || F % WG_TILE_F != 0 || H > 4096 || F > 4096) return false;
  if (n_op < 1 || n_op > 2) return false;
  s->tiles_h = (int)((H + WG_TILE_H - 1) / WG_TILE_H);
  s->tiles_f = (int)(F / WG_TILE_F);
  const int64_t per_slab = (int64_t)s->tiles_h * s->tiles_f * n_op;
  int64_t slabs = (WG_TARGET_BLOCKS + per_slab - 1) / per_slab;
  const int64_t most = (n + WG_MIN_SLAB_ROWS - 1) / WG_MIN_SLAB_ROWS;
  if (slabs > most) slabs = most;
  const int64_t rows = (n + slabs - 1) / slabs;
  s->slab_rows = (rows + 3) / 4 * 4;                 // a matrix instruction takes four rows
  s->slabs = (n + s->slab_rows - 1) / s->slab_rows;
  return true;
}

// Four adjacent elements at byte `at`, the first `valid` of them (whole quads where VEC); the others are zeros.
template <bool VEC>
__device__ __forceinline__ wg_quad wg_load(hc_buffer b, uint32_t at, int valid) {
  constexpr uint32_t NOWHERE = 0xfffffff0u;
  if (valid <= 0) at = NOWHERE;
  if constexpr (VEC) {
    return __builtin_bit_cast(wg_quad, __builtin_amdgcn_raw_buffer_load_b128(b, at, 0, 0));
  } else {
    wg_quad v;
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = __builtin_amdgcn_raw_buffer_load_b32(b, q < valid ? at + 4u * q : NOWHERE, 0, 0);
    return v;
  }
}

template <bool VEC>
__global__ __launch_bounds__(HC_BLOCK) void wg_partial(const float *__restrict__ g, const float *__restrict__ x0,
                                                        const float *__restrict__ x1, float *__restrict__ part,
                                                        float *__restrict__ part_sum, int64_t n, int H, int F,
                                                        int per_slab, WgShape sh) {
  constexpr int BM = WG_TILE_H, BN = WG_TILE_F, BK = WG_PIECE;
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16, LDG = BM + 16, LDX = BN + 16;
  constexpr int QG = BM / 4, QX = BN / 4, NG = BK * QG / HC_BLOCK, NX = BK * QX / HC_BLOCK;
  __shared__ __attribute__((aligned(16))) float sg[2][BK * LDG], sx[2][BK * LDX];
  // blocks of one slab lie side by side: they read the same rows
  const int64_t b = hc_xcd_block<16>(blockIdx.x, gridDim.x);
  const int64_t slab = b / per_slab;
  const int in_slab = (int)(b % per_slab), tiles = sh.tiles_h * sh.tiles_f;
  const int op = in_slab / tiles, tile = in_slab % tiles;
  const int f0 = tile % sh.tiles_f * BN, h0 = tile / sh.tiles_f * BM;
  const float *__restrict__ x = op == 0 ? x0 : x1;
  const int64_t lo = slab * sh.slab_rows, hi = lo + sh.slab_rows < n ? lo + sh.slab_rows : n;
  const int t = (int)threadIdx.x, lane = hc_lane(), wave = hc_wave_in_block();
  const int wm = (wave & 1) * WM, wn = (wave >> 1) * WN;
  const int l16 = lane & 15, k4 = lane >> 4;
  const bool sums = part_sum != nullptr && op == 0 && f0 == 0;       // this block adds up g's columns, too
  float col_sum = 0.f;
  uint32_t at_g[NG], at_x[NX];
  int valid_g[NG];
#pragma unroll
  for (int i = 0; i < NG; ++i) {
    const int f = t + i * HC_BLOCK;
    at_g[i] = (uint32_t)(f / QG * H + h0 + f % QG * 4) * 4u;
    valid_g[i] = H - (h0 + f % QG * 4);
  }
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int f = t + i * HC_BLOCK;
    at_x[i] = (uint32_t)(f / QX * F + f0 + f % QX * 4) * 4u;
  }
  wg_quad rg[NG], rx[NX];
  const auto load = [&](int64_t r) {
    const uint32_t rows = (uint32_t)(hi - r < BK ? hi - r : BK);
    const hc_buffer bg = hc_make_buffer(g + r * H, rows * (uint32_t)H * 4u), bx = hc_make_buffer(x + r * F, rows * (uint32_t)F * 4u);
#pragma unroll
    for (int i = 0; i < NG; ++i) rg[i] = wg_load<VEC>(bg, at_g[i], valid_g[i]);
#pragma unroll
    for (int i = 0; i < NX; ++i) rx[i] = wg_load<VEC>(bx, at_x[i], 4);
  };
  const auto stage = [&](int s) {
#pragma unroll
    for (int i = 0; i < NG; ++i) {
      const int f = t + i * HC_BLOCK;
      *reinterpret_cast<wg_quad *>(&sg[s][f / QG * LDG + f % QG * 4]) = rg[i];
    }
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int f = t + i * HC_BLOCK;
      *reinterpret_cast<wg_quad *>(&sx[s][f / QX * LDX + f % QX * 4]) = rx[i];
    }
  };
  wg_acc acc[TM][TN], sum[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j] = wg_acc{0.f, 0.f, 0.f, 0.f};
  static_assert(WG_CHAIN_ROWS % BK == 0, "whole pieces per chain");
  const auto end_chain = [&]() {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        sum[i][j] += acc[i][j];
        acc[i][j] = wg_acc{0.f, 0.f, 0.f, 0.f};
      }
  };
  const auto step = [&](int s, int k) {
    float u[TM], v[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) u[i] = sg[s][(k + k4) * LDG + wm + i * 16 + l16];
#pragma unroll
    for (int j = 0; j < TN; ++j) v[j] = sx[s][(k + k4) * LDX + wn + j * 16 + l16];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j], u[i], acc[i][j], 0, 0, 0);
  };
  // one column per lane, a quarter of the piece's rows per wave (rows behind the slab are zeros)
  const auto add_columns = [&](int s) {
#pragma unroll
    for (int k = 0; k < BK / HC_WAVES_PER_BLOCK; ++k) col_sum += sg[s][(wave * (BK / HC_WAVES_PER_BLOCK) + k) * LDG + lane];
  };
  load(lo);
  stage(0);
  int s = 0;
  int64_t r = lo;
  for (; r + BK < hi; r += BK) {
    __syncthreads();
    load(r + BK);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < BK; k += 4) step(s, k);
    if (sums) add_columns(s);
    __builtin_amdgcn_sched_barrier(0);
    s ^= 1;
    stage(s);
    if (((uint32_t)(r - lo) + BK) % WG_CHAIN_ROWS == 0) end_chain();
  }
  __syncthreads();
  for (int k = 0; k < (int)(hi - r); k += 4) step(s, k);           // the last piece: 1 to WG_PIECE rows
  if (sums) {
    add_columns(s);
    part_sum[(slab * HC_WAVES_PER_BLOCK + wave) * (sh.tiles_h * BM) + h0 + lane] = col_sum;
  }
  end_chain();
  // partial tile of this block, tiles ordered (operand, tile, slab)
  float *o = part + ((int64_t)in_slab * sh.slabs + slab) * (BM * BN);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *reinterpret_cast<wg_acc *>(o + (wm + i * 16 + l16) * BN + wn + j * 16 + 4 * k4) = sum[i][j];
}

// dW[op][h][f]: a quarter of the slabs per wave, in slab order, then the quarters in order.  Four columns per lane;
// four waves share them because a lane's loads, one per slab, are what the launch waits for (89 000 rows, 64 x 64, two
// operands, 512 slabs: both launches 44 us with one wave's chain, 30 with four).
__global__ __launch_bounds__(HC_BLOCK) void wg_reduce(const float *__restrict__ part, float *__restrict__ dw0,
                                                       float *__restrict__ dw1, const float *__restrict__ part_sum,
                                                       float *__restrict__ dsum, int n_op, int H, int F, WgShape sh) {
  constexpr int Q = WG_TILE_F / 4, FLIGHT = 8;         // float4 groups per tile row
  __shared__ float4 s_part[3][HC_WAVE];
  const int lane = hc_lane(), wave = hc_wave_in_block();
  if ((int)blockIdx.y == n_op) {                       // the sums of g's columns, one column per lane
    const int c = (int)blockIdx.x * HC_WAVE + lane;
    if ((int)blockIdx.x >= sh.tiles_h) return;
    float v = 0.f;
    for (int64_t i = sh.slabs * wave; i < sh.slabs * (wave + 1); ++i) v += part_sum[i * (sh.tiles_h * WG_TILE_H) + c];
    if (wave > 0) s_part[wave - 1][lane].x = v;
    __syncthreads();
    if (wave > 0 || c >= H) return;
    for (int w = 0; w < 3; ++w) v += s_part[w][lane].x;
    dsum[c] = v;
    return;
  }
  const int64_t t = (int64_t)blockIdx.x * HC_WAVE + lane;          // the grid covers whole tiles
  const int q = (int)(t % Q), hl = (int)(t / Q % WG_TILE_H), tile = (int)(t / (Q * WG_TILE_H));
  const int op = (int)blockIdx.y;
  constexpr int64_t TILE = WG_TILE_H * WG_TILE_F;
  const float *p = part + ((int64_t)op * sh.tiles_h * sh.tiles_f + tile) * sh.slabs * TILE + (int64_t)hl * WG_TILE_F + 4 * q;
  int64_t k = sh.slabs * wave / 4;
  const int64_t end = sh.slabs * (wave + 1) / 4;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  const auto plus = [&](const float4 &v) { s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w; };
  for (; k + FLIGHT <= end; k += FLIGHT) {
    float4 v[FLIGHT];
#pragma unroll
    for (int j = 0; j < FLIGHT; ++j) v[j] = *reinterpret_cast<const float4 *>(p + (k + j) * TILE);
    // pairs, pairs of pairs, then the sum so far: an eighth of the additions in one chain
#pragma unroll
    for (int w = FLIGHT / 2; w > 0; w /= 2)
#pragma unroll
      for (int j = 0; j < w; ++j) {
        v[j].x += v[j + w].x; v[j].y += v[j + w].y; v[j].z += v[j + w].z; v[j].w += v[j + w].w;
      }
    plus(v[0]);
  }
  for (; k < end; ++k) plus(*reinterpret_cast<const float4 *>(p + k * TILE));
  if (wave > 0) s_part[wave - 1][lane] = s;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < 3; ++w) plus(s_part[w][lane]);
  const int h = tile / sh.tiles_f * WG_TILE_H + hl, f = tile % sh.tiles_f * WG_TILE_F + 4 * q;
  if (h >= H) return;
  *reinterpret_cast<float4 *>((op == 0 ? dw0 : dw1) + (int64_t)h * F + f) = s;
}

}  // namespace

static_assert(WG_TILE_H == HC_WAVE, "one column of a tile per lane");

// Bytes of the partial tiles, and behind them of the partial sums of g's columns.
static size_t wg_tile_bytes(const WgShape &sh, int n_op) {
  return (size_t)n_op * sh.tiles_h * sh.tiles_f * sh.slabs * WG_TILE_H * WG_TILE_F * sizeof(float);
}
static size_t wg_sum_bytes(const WgShape &sh) { return (size_t)sh.slabs * HC_WAVES_PER_BLOCK * sh.tiles_h * WG_TILE_H * sizeof(float); }

static int wg_run(const float *g, const float *x0, const float *x1, int64_t n, int64_t H, int64_t F, float *dw0, float *dw1,
                  float *dsum, const WgShape &sh, int n_op, void *workspace, size_t workspace_bytes, hipStream_t st) {
  if (!workspace || workspace_bytes < wg_tile_bytes(sh, n_op) + (dsum ? wg_sum_bytes(sh) : 0) ||
      reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
    return HC_EWORKSPACE;
  if (reinterpret_cast<uintptr_t>(dw0) % 16 != 0 || (dw1 && reinterpret_cast<uintptr_t>(dw1) % 16 != 0))
    return HC_EINVAL;
  float *part = static_cast<float *>(workspace);
  float *part_sum = dsum ? part + wg_tile_bytes(sh, n_op) / sizeof(float) : nullptr;
  const int per_slab = sh.tiles_h * sh.tiles_f * n_op;
  const int64_t blocks = sh.slabs * per_slab;
  if (!hc_grid_ok(blocks)) return HC_EUNSUPPORTED;
  const bool vec = H % 4 == 0 &&
                   (reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(x0) | reinterpret_cast<uintptr_t>(x1)) % 16 == 0;
  const auto kernel = vec ? wg_partial<true> : wg_partial<false>;
  kernel<<<dim3((unsigned)blocks), dim3(HC_BLOCK), 0, st>>>(g, x0, x1, part, part_sum, n, (int)H, (int)F, per_slab, sh);
  const int64_t quads = (int64_t)sh.tiles_h * sh.tiles_f * WG_TILE_H * (WG_TILE_F / 4);
  wg_reduce<<<dim3((unsigned)(quads / HC_WAVE), (unsigned)(n_op + (dsum ? 1 : 0))), dim3(HC_BLOCK), 0, st>>>(
      part, dw0, dw1, part_sum, dsum, n_op, (int)H, (int)F, sh);
  return hc_launch_status();
}

extern "C" size_t hc_weight_grad_workspace_bytes(int64_t n, int64_t H, int64_t F, int n_operands) {
  WgShape sh;
  if (H % WG_TILE_H != 0 || !wg_shape(n, H, F, n_operands, &sh)) return 0;
  return hc_align_up(wg_tile_bytes(sh, n_operands), 256);
}

extern "C" int hc_weight_grad(const float *g, const float *x0, const float *x1, int64_t n, int64_t H, int64_t F,
                              float *dw0, float *dw1, void *workspace, size_t workspace_bytes, void *stream) {
  HC_REQUIRE(g && x0 && dw0 && (x1 == nullptr) == (dw1 == nullptr));
  const int n_op = x1 != nullptr ? 2 : 1;
  WgShape sh;
  if (H % WG_TILE_H != 0 || !wg_shape(n, H, F, n_op, &sh)) return n >= 1 && H >= 1 && F >= 1 ? HC_EUNSUPPORTED : HC_EINVAL;
  return wg_run(g, x0, x1, n, H, F, dw0, dw1, nullptr, sh, n_op, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" size_t hc_linear_grad_workspace_bytes(int64_t n, int64_t H, int64_t F, int n_operands) {
  WgShape sh;
  if (!wg_shape(n, H, F, n_operands, &sh)) return 0;
  return hc_align_up(wg_tile_bytes(sh, n_operands) + wg_sum_bytes(sh), 256);
}

extern "C" int hc_linear_grad(const float *g, const float *x0, const float *x1, int64_t n, int64_t H, int64_t F,
                              float *dw0, float *dw1, float *dbias, void *workspace, size_t workspace_bytes,
                              void *stream) {
  HC_REQUIRE(g && x0 && dw0 && (x1 == nullptr) == (dw1 == nullptr));
  const int n_op = x1 != nullptr ? 2 : 1;
  WgShape sh;
  if (!wg_shape(n, H, F, n_op, &sh)) return n >= 1 && H >= 1 && F >= 1 ? HC_EUNSUPPORTED : HC_EINVAL;
  return wg_run(g, x0, x1, n, H, F, dw0, dw1, dbias, sh, n_op, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
