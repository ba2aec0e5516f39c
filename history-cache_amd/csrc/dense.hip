// The dense half of a layer: out[M, N] = A0 op(W0) [+ A1 op(W1)] [+ add] [+ bias], fp32 in and out, M = rows of a sampled
// layer (thousands to hundreds of thousands), N and K a few hundred.  What `lin_l(out) + lin_r(x[:n])` and its input
// gradients are (/root/reference/hiscache/history_model.py:94-98): forward with W as torch.nn.Linear keeps it, [N, K];
// backward with the same matrix read as [K, N].
//
// What bounds it: the matrix pipes (v_mfma_f32_16x16x4_f32; a loop of nothing else reaches 148 TFLOP/s with two waves per
// SIMD and 128 with four).  They are busy 78% of a block's time; launch, first pieces and the last round of tiles take
// the rest.  Measured, two products and the bias, library GEMMs + bias add / this: 190 000 rows, K = 100, N = 256
// 363 / 209 us (93 TFLOP/s); 55 000, 128, 256 115 / 70; 36 000, 256, 256 102 / 84 (112); 8 700, 256, 256 40 / 32; 1 000, 256, 172
// 22 / 8.  One product with W as [K, N]: 55 000, 256, 128 80 / 39; 8 700, 256, 256 21 / 19.  Tiles of 128 x 128, 128 x 64
// and 64 x 128, pieces of 16 and 64 columns, v_mfma_f32_32x32x2_f32 and two or three blocks per compute unit instead of
// four: 2 to 30% slower where the rows are few, no faster where they are many.
//
// Loads of A, loads of W and the way out are 16 bytes wide wherever their own width and alignment allow it: the gradient of
// 47 classes is read by single elements, W and the result are not.  One product with W as [K, N], inner size 47, everything
// by single elements / only A: 60 000 rows, N = 256 50 / 26 us; 20 000, 768 53 / 26; 1 000, 256 4.2 / 3.4.
//
// A block of four waves stages K in pieces through two LDS buffers: the loads of a piece are issued in front of the
// matrix instructions of the one before it (kept there by a scheduling barrier: left alone, the compiler moves them
// behind, and every wave waits for them).  Rows and columns behind the matrices are read
// through buffer descriptors, which answer with zeros, so that no load is in a branch.  Staged rows are two words longer
// than a piece: the 16 rows x 2 columns that half a wave reads at once then lie in 32 banks.
//
// The operands are handed to the instruction in exchanged roles (W as its rows), so that a lane ends with four adjacent
// columns of one row of the result, one 16-byte store:
//   A operand (16 x 4): W's column n0 + l % 16 at k + l / 16        B operand (4 x 16): A's row m0 + l % 16 at k + l / 16
//   D (16 x 16, 4 values per lane): row of `out` m0 + l % 16, columns n0 + 4 (l / 16) .. + 3
//
// In evaluation the layer's batch normalisation and ReLU take the tile on its way out (NORM): a pass over the result and
// its way through memory less: an evaluation batch of 4 000 seeds, 256 channels, two such layers, 774 us as two launches
// each, 681 as one.
//
// Summation order: a product by itself is two chains, the even and the odd steps of four columns, each summed from zero in
// ascending k, and added at the end; of two products each is one chain, and the second is added to the first; then `add`, then
// the bias -- whatever the tile, so a row's result does not depend on how many rows there are.  Two chains because the library
// has them where the rows are few: error against 64 bits of 1 000 rows, inner size 256, one chain 2.9e-7, two 2.1e-7 (library
// 2.1); 172 2.4, 1.7 (1.7); 47 1.2, 0.9 (0.9).  With two products the library has one chain as well.  Held to the registers of
// four waves per SIMD the 64 x 64 tile is a little faster with two than it was with one: 55 000 rows, 256 to 128 36.7 / 36.3 us.
#include "hc_common.h"

namespace {

typedef float lin_acc __attribute__((ext_vector_type(4)));

struct LinArgs {
  const float *a0, *a1, *w0, *w1, *bias, *add;
  float *out;
  int64_t M;
  int N, K, tiles_n;
  bool whole;                                  // four adjacent columns of the result, `add` and the bias lie on 16 bytes
  const float *mean, *var, *gamma, *beta;      // batch normalisation and ReLU behind the bias (NORM)
  float eps;
};

typedef uint32_t lin_quad __attribute__((ext_vector_type(4)));

// Four adjacent elements of a row that starts `row` bytes into the buffer; those behind `end` are zeros.
template <bool VEC>
__device__ __forceinline__ lin_quad lin_load(hc_buffer b, uint32_t row, int at, int end) {
  constexpr uint32_t NOWHERE = 0xfffffff0u;
  if constexpr (VEC) {
    return __builtin_bit_cast(lin_quad, __builtin_amdgcn_raw_buffer_load_b128(b, at < end ? row + (uint32_t)at * 4u : NOWHERE, 0, 0));
  } else {
    lin_quad v;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = __builtin_amdgcn_raw_buffer_load_b32(b, at + q < end ? row + (uint32_t)(at + q) * 4u : NOWHERE, 0, 0);
    return v;
  }
}

template <int BM, int BN, int BK, bool KN, bool VEC_A, bool VEC_W, bool TWO, bool NORM>
__global__ __launch_bounds__(HC_BLOCK, BM == 64 ? 4 : 1) void lin_tile(LinArgs a) {
  constexpr int WM = BM / 2, WN = BN / 2, TM = WM / 16, TN = WN / 16;
  constexpr int LDA = BK + 2, LDW = KN ? BN + 16 : BK + 2;
  constexpr int QA = BK / 4, QW = KN ? BN / 4 : BK / 4;                  // four-element pieces of a staged row
  constexpr int NA = BM * BK / 4 / HC_BLOCK, NW = BN * BK / 4 / HC_BLOCK;
  __shared__ __attribute__((aligned(16))) float sa[2][BM * LDA];
  __shared__ __attribute__((aligned(16))) float sw[2][KN ? BK * LDW : BN * LDW];
  __shared__ __attribute__((aligned(16))) float sn[NORM ? 5 : 1][NORM ? BN : 1];
  const int64_t tile = hc_xcd_block<16>(blockIdx.x, gridDim.x);
  const int64_t m0 = tile / a.tiles_n * BM;
  const int n0 = (int)(tile % a.tiles_n) * BN;
  const int t = (int)threadIdx.x, lane = hc_lane(), wave = hc_wave_in_block();
  const int wm = (wave & 1) * WM, wn = (wave >> 1) * WN;
  const int l16 = lane & 15, g = lane >> 4;
  const int rows_a = (int)(a.M - m0 < BM ? a.M - m0 : BM), rows_w = a.N - n0 < BN ? a.N - n0 : BN;
  const uint32_t bytes_a = (uint32_t)(rows_a * a.K) * 4u;
  const uint32_t bytes_w = KN ? (uint32_t)a.K * (uint32_t)a.N * 4u : (uint32_t)rows_w * (uint32_t)a.K * 4u;
  const int64_t at_a = m0 * a.K, at_w = KN ? 0 : (int64_t)n0 * a.K;
  const float *pa = a.a0 + at_a, *pw = a.w0 + at_w;
  lin_quad ra[NA], rw[NW];
  const auto load = [&](int k0) {
    const hc_buffer ba = hc_make_buffer(pa, bytes_a), bw = hc_make_buffer(pw, bytes_w);
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int f = t + i * HC_BLOCK;
      ra[i] = lin_load<VEC_A>(ba, (uint32_t)(f / QA) * (uint32_t)a.K * 4u, k0 + f % QA * 4, a.K);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int f = t + i * HC_BLOCK;
      if constexpr (KN) rw[i] = lin_load<VEC_W>(bw, (uint32_t)(k0 + f / QW) * (uint32_t)a.N * 4u, n0 + f % QW * 4, a.N);
      else rw[i] = lin_load<VEC_W>(bw, (uint32_t)(f / QW) * (uint32_t)a.K * 4u, k0 + f % QW * 4, a.K);
    }
  };
  const auto put = [&](float *at, const lin_quad &v) {
    typedef uint32_t pair __attribute__((ext_vector_type(2)));
    reinterpret_cast<pair *>(at)[0] = pair{v[0], v[1]};
    reinterpret_cast<pair *>(at)[1] = pair{v[2], v[3]};
  };
  const auto stage = [&](int b) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int f = t + i * HC_BLOCK;
      put(&sa[b][f / QA * LDA + f % QA * 4], ra[i]);
    }
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int f = t + i * HC_BLOCK;
      if constexpr (KN) *reinterpret_cast<lin_quad *>(&sw[b][f / QW * LDW + f % QW * 4]) = rw[i];
      else put(&sw[b][f / QW * LDW + f % QW * 4], rw[i]);
    }
  };
  constexpr int CHAINS = TWO ? 1 : 2;
  static_assert(BK % 8 == 0, "a piece starts with the first chain");
  lin_acc chain[CHAINS][TM][TN], sum[TWO ? TM : 1][TWO ? TN : 1];
  auto &acc = chain[0], &other = chain[CHAINS - 1];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = other[i][j] = lin_acc{0.f, 0.f, 0.f, 0.f};
  const auto step = [&](lin_acc (&to)[TM][TN], int b, int k) {
    float x[TM], y[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) x[i] = sa[b][(wm + i * 16 + l16) * LDA + k + g];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      y[j] = KN ? sw[b][(k + g) * LDW + wn + j * 16 + l16] : sw[b][(wn + j * 16 + l16) * LDW + k + g];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(y[j], x[i], to[i][j], 0, 0, 0);
  };
  load(0);
  if constexpr (NORM) {
    // bias, mean, 1 / sqrt(var + eps), gamma and beta of the tile's columns, a square root and a division per column
    static_assert(BN <= HC_BLOCK, "one thread per column");
    if (t < BN) {
      const int n = n0 + t < a.N ? n0 + t : a.N - 1;
      sn[0][t] = a.bias != nullptr ? a.bias[n] : 0.f;
      sn[1][t] = a.mean[n];
      sn[2][t] = 1.0f / sqrtf(a.var[n] + a.eps);
      sn[3][t] = a.gamma != nullptr ? a.gamma[n] : 1.f;
      sn[4][t] = a.beta != nullptr ? a.beta[n] : 0.f;
    }
  }
  stage(0);
  int b = 0;
  for (int p = 0; p < (TWO ? 2 : 1); ++p) {
    int k0 = 0;
    for (; k0 + BK < a.K; k0 += BK) {
      __syncthreads();
      load(k0 + BK);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < BK; k += 8) {
        step(acc, b, k);
        step(other, b, k + 4);
      }
      __builtin_amdgcn_sched_barrier(0);
      b ^= 1;
      stage(b);
    }
    // the product's last piece, of 1 to BK columns, while the second product's first is on its way
    __syncthreads();
    if (TWO && p == 0) {
      pa = a.a1 + at_a;
      pw = a.w1 + at_w;
      load(0);
    }
    __builtin_amdgcn_sched_barrier(0);
    const int left = a.K - k0;
    if (left == BK) {
#pragma unroll
      for (int k = 0; k < BK; k += 8) {
        step(acc, b, k);
        step(other, b, k + 4);
      }
    } else {
      int k = 0;
      for (; k + 4 < left; k += 8) {
        step(acc, b, k);
        step(other, b, k + 4);
      }
      if (k < left) step(acc, b, k);
    }
    b ^= 1;
    if (TWO && p == 0) stage(b);
    if constexpr (!TWO) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] += other[i][j];
    } else {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          sum[i][j] = p == 0 ? acc[i][j] : sum[i][j] + acc[i][j];
          acc[i][j] = lin_acc{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  // lane l holds columns 4 (l / 16) .. + 3 of row l % 16 of every 16 x 16 piece
  if constexpr (TWO) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = sum[i][j];
  }
  const auto plus = [&](const float *__restrict__ add, int64_t row_step) {
    lin_acc v[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      int64_t m = m0 + wm + i * 16 + l16;
      m = m < a.M ? m : a.M - 1;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = n0 + wn + j * 16 + 4 * g;
        const float *o = add + m * row_step;
        if (a.whole) {
          v[i][j] = *reinterpret_cast<const lin_acc *>(o + (n < a.N ? n : a.N - 4));
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[i][j][q] = o[n + q < a.N ? n + q : a.N - 1];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] += v[i][j];
  };
  if constexpr (NORM) {
    // the same expression as the separate pass (bn_eval): same bits; NaN stays NaN
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      lin_acc c[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) c[q] = *reinterpret_cast<const lin_acc *>(&sn[q][wn + j * 16 + 4 * g]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float v = (((acc[i][j][q] + c[0][q]) - c[1][q]) * c[2][q]) * c[3][q] + c[4][q];
          acc[i][j][q] = v < 0.f ? 0.f : v;
        }
    }
  } else {
    if (a.add != nullptr) plus(a.add, a.N);
    if (a.bias != nullptr) plus(a.bias, 0);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int64_t m = m0 + wm + i * 16 + l16;
    if (m >= a.M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + j * 16 + 4 * g;
      float *o = a.out + m * a.N + n;
      if (a.whole) {
        if (n < a.N) *reinterpret_cast<lin_acc *>(o) = acc[i][j];
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < a.N) o[q] = acc[i][j][q];
      }
    }
  }
}

template <int BM, int BN, int BK>
int lin_launch(LinArgs a, bool kn, bool vec_a, bool vec_w, hipStream_t st) {
  a.tiles_n = (a.N + BN - 1) / BN;
  const int64_t blocks = (a.M + BM - 1) / BM * a.tiles_n;
  if (!hc_grid_ok(blocks)) return HC_EUNSUPPORTED;
  const dim3 grid((unsigned)blocks), block(HC_BLOCK);
#define HC_LIN(KN, VEC_A, VEC_W)                                                                               \
  {                                                                                                            \
    if (a.a1 != nullptr) lin_tile<BM, BN, BK, KN, VEC_A, VEC_W, true, NORM><<<grid, block, 0, st>>>(a);        \
    else lin_tile<BM, BN, BK, KN, VEC_A, VEC_W, false, NORM><<<grid, block, 0, st>>>(a);                       \
  }
  constexpr bool NORM = false;
  if (a.mean != nullptr) {
    constexpr bool NORM = true;
    if (vec_a && vec_w) HC_LIN(false, true, true)
    else HC_LIN(false, false, false)
  } else if (kn && vec_a && vec_w) HC_LIN(true, true, true)
  else if (kn && vec_w) HC_LIN(true, false, true)
  else if (kn) HC_LIN(true, false, false)
  else if (vec_a && vec_w) HC_LIN(false, true, true)
  else HC_LIN(false, false, false)
#undef HC_LIN
  return hc_launch_status();
}

// Up to this many results tiles of 64 x 64 leave more than half of the chip idle; tiles of 32 x 32 then fill it, and their
// deep pieces (128 columns) take fewer round trips.  64 x 64 / 32 x 32: 1 000 rows, K = 256, N = 172 13.5 / 8.3 us; 4 000, 256,
// 47 14.4 / 9.3; 6 000, 128, 128 9.9 / 10.4; 36 000, 256, 256 84 / 140.
constexpr int64_t LIN_SMALL = (int64_t)1 << 19;
// Up to this many columns tiles of 64 x 64 are half or more padding, and pieces of 64 columns leave room for another block per
// compute unit.  Two products and the bias, 64 x 64 / 32 x 32 with pieces of 64: 60 000 rows, K = 768, N = 10 108 / 72 us (library
// GEMMs 80); 200 000, 256, 32 118 / 89 (108); 30 000, 256, 32 22 / 15 (26); 1 000, 64, 10 with pieces of 128 4.4 / 3.5.
constexpr int LIN_NARROW = 32;
constexpr int64_t LIN_MAX = (int64_t)1 << 20;      // N and K; a tile's rows and W are addressed by 32-bit offsets
constexpr int LIN_PIECE = 128;                     // longest piece of K

}  // namespace

static int lin_run(LinArgs a, bool kn, hipStream_t st) {
  HC_REQUIRE(a.a0 && a.w0 && a.out && (a.a1 == nullptr) == (a.w1 == nullptr) && a.M >= 1);
  const auto on16 = [](const float *p, const float *q, const float *r) {
    return (reinterpret_cast<uintptr_t>(p) | reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(r)) % 16 == 0;
  };
  const bool vec_a = a.K % 4 == 0 && on16(a.a0, a.a1, nullptr);
  const bool vec_w = (kn ? a.N : a.K) % 4 == 0 && on16(a.w0, a.w1, nullptr);
  a.whole = a.N % 4 == 0 && on16(a.out, a.add, a.bias);
  if (a.N <= LIN_NARROW) return lin_launch<32, 32, 64>(a, kn, vec_a, vec_w, st);
  if (a.M <= LIN_SMALL / a.N) return lin_launch<32, 32, LIN_PIECE>(a, kn, vec_a, vec_w, st);
  return lin_launch<64, 64, 32>(a, kn, vec_a, vec_w, st);
}

// N and K as the kernel takes them.  W [K, N] is read up to one piece (LIN_PIECE rows at most) behind its last row: their
// offsets must not come round to W's first rows, and the offset that stands for no element must lie behind its last.
static int lin_widths(int64_t N, int64_t K) {
  HC_REQUIRE(N >= 1 && K >= 1);
  return N > LIN_MAX || K > LIN_MAX || (K + LIN_PIECE) * N >= (int64_t)1 << 30 ? HC_EUNSUPPORTED : HC_OK;
}

extern "C" int hc_linear(const float *a0, const float *w0, const float *a1, const float *w1, int w_is_kn,
                         const float *bias, const float *add, float *out, int64_t M, int64_t N, int64_t K,
                         void *stream) {
  if (const int rc = lin_widths(N, K)) return rc;
  const LinArgs a{a0, a1, w0, w1, bias, add, out, M, (int)N, (int)K, 0, false, nullptr, nullptr, nullptr, nullptr, 0.f};
  return lin_run(a, w_is_kn != 0, static_cast<hipStream_t>(stream));
}

extern "C" int hc_linear_bn_relu(const float *a0, const float *w0, const float *a1, const float *w1, const float *bias,
                                 const float *gamma, const float *beta, const float *running_mean,
                                 const float *running_var, float eps, float *out, int64_t M, int64_t N, int64_t K,
                                 void *stream) {
  if (const int rc = lin_widths(N, K)) return rc;
  HC_REQUIRE(running_mean && running_var);
  const LinArgs a{a0, a1, w0, w1, bias, nullptr, out, M, (int)N, (int)K, 0, false, running_mean, running_var, gamma, beta, eps};
  return lin_run(a, false, static_cast<hipStream_t>(stream));
}
