// The gradient of the edge weights: edge_grad[j, h] = <g[r, h, :], vin[idx[j], h, :]> for the edges of the first R
// rows, 0 for edges of history rows and for the slots behind the last row, as in the reference
// (/root/reference/src/cpp/src/history_aggr.cu:258-267, :329-397).
//
// One wave per 64 consecutive edge slots, whatever rows they belong to (a row of thousands of edges is shared by
// many waves).  The lanes are dealt to the heads: LPH = a power of two of them per head, several heads side by
// side; wider heads and further heads are walked in steps.  UNROLL edges are in flight at a time; a head's lanes
// are summed with row permutations and lane swaps of the vector unit, which leave the LDS out.
//
// What bounds it: 1 M edges of four heads of 32 fp32 columns move 1 GB through the L1s.  With shuffles through the
// LDS (four per edge) and a bisection of the row offsets in front of every wave it took 131 us, now 105.  (Widths
// off a multiple of 64 were walked by one wave per row, edge after edge: a long row took a microsecond an edge.)
#include "hc_common.h"
#include "tr_shared.h"

namespace {

struct EdgeGradArgs {
  const int64_t *ptr, *idx;
  const float *g;
  const int64_t *hmap;
  const void *vin;
  float *edge_grad;
  int64_t E, R;
  int H, fh;        // heads, columns per head
  int lph_bits;     // log2 of the lanes per head
};

// Sum over the 2^bits lanes of an aligned group; every lane of the group ends with it.  The partners are at
// distance 1, 2, 4 and 8 (mirrored halves: the lanes of a quad or an eighth already agree), 16 and 32.
__device__ __forceinline__ float eg_group_sum(float v, int bits) {
#define HC_EG_DPP(ctrl) \
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl, 0xf, 0xf, true))
  if (bits > 0) HC_EG_DPP(0xB1);      // quad_perm [1, 0, 3, 2]
  if (bits > 1) HC_EG_DPP(0x4E);      // quad_perm [2, 3, 0, 1]
  if (bits > 2) HC_EG_DPP(0x141);     // row_half_mirror
  if (bits > 3) HC_EG_DPP(0x140);     // row_mirror
#undef HC_EG_DPP
  if (bits > 4) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  if (bits > 5) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
  }
  return v;
}

template <typename T, int VEC, int UNROLL>
__global__ __launch_bounds__(HC_BLOCK) void edge_grad_rows(EdgeGradArgs a) {
  const int lane = hc_lane();
  const int64_t base = ((int64_t)blockIdx.x * HC_WAVES_PER_BLOCK + hc_wave_in_block()) * HC_WAVE;
  if (base >= a.E) return;
  const int n = a.E - base < HC_WAVE ? (int)(a.E - base) : HC_WAVE;
  // rows of the first and the last slot, then of every lane's own
  int my_row = -1;
  int64_t my_id = 0;
  if (a.R > 0 && a.ptr[0] <= base + n - 1) {
    const int64_t lo = tr_row_of_wave(a.ptr, a.R, base, lane), hi = tr_row_of_wave(a.ptr, a.R, base + n - 1, lane);
    if (lane < n) {
      const int64_t e = base + lane;
      const int64_t r = tr_row_of(a.ptr, lo, hi, e);
      if (r < a.R && a.ptr[r] <= e && (a.hmap == nullptr || a.hmap[r] == -1)) {
        my_row = (int)r;
        my_id = a.idx[e];
      }
    }
  }
  unsigned long long todo = __ballot(my_row >= 0);
  const int lph = 1 << a.lph_bits;
  const int side = HC_WAVE >> a.lph_bits;               // heads side by side
  const int sub = lane & (lph - 1);
  const int64_t row_elems = (int64_t)a.H * a.fh;
  float my_out = 0.0f;
  while (todo != 0ull) {
    int pos[UNROLL];
    int64_t xb[UNROLL], gb[UNROLL];                     // addresses of the edges' rows
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      pos[u] = todo != 0ull ? __builtin_ctzll(todo) : pos[u > 0 ? u - 1 : 0];     // behind the end: the last one again
      todo &= todo - 1ull;
      xb[u] = reinterpret_cast<int64_t>(static_cast<const T *>(a.vin) + hc_readlane64(my_id, pos[u]) * row_elems);
      gb[u] = reinterpret_cast<int64_t>(a.g + (int64_t)__builtin_amdgcn_readlane(my_row, pos[u]) * row_elems);
    }
    for (int h0 = 0; h0 < a.H; h0 += side) {
      const int head = h0 + (lane >> a.lph_bits);
      float part[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) part[u] = 0.0f;
      for (int c0 = 0; c0 < a.fh; c0 += lph * VEC) {
        const int c = c0 + sub * VEC;
        if (c < a.fh && head < a.H) {
          const uint32_t off = (uint32_t)(head * a.fh + c);
          typename hc_piece<T, VEC>::raw_t x[UNROLL];
          typename hc_piece<float, VEC>::raw_t gr[UNROLL];
#pragma unroll
          for (int u = 0; u < UNROLL; ++u) {
            x[u] = hc_piece<T, VEC>::template load<false>(xb[u], off * (uint32_t)sizeof(T));
            gr[u] = hc_piece<float, VEC>::template load<false>(gb[u], off * 4u);
          }
#pragma unroll
          for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int i = 0; i < VEC; ++i)
              part[u] = __fmaf_rn(hc_piece<float, VEC>::widen(gr[u], i), hc_piece<T, VEC>::widen(x[u], i), part[u]);
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const float sum = eg_group_sum(part[u], a.lph_bits);
        if (a.H == 1) my_out = lane == pos[u] ? hc_readlane_f(sum, 0) : my_out;   // lane 0 lies in the head's group
        else if (sub == 0 && head < a.H) a.edge_grad[(base + pos[u]) * a.H + head] = sum;
      }
    }
  }
  if (a.H == 1) {
    if (lane < n) a.edge_grad[base + lane] = my_out;
  } else if (lane < n && my_row < 0) {
    float *__restrict__ o = a.edge_grad + (base + lane) * a.H;
    for (int h = 0; h < a.H; ++h) o[h] = 0.0f;
  }
}

// Elements per lane and load: the widest that a head's width and the pointers allow, halved while the heads still
// fit the wave side by side (all lanes busy rather than wide loads by a few).
template <typename T>
int eg_launch(EdgeGradArgs &a, hipStream_t st) {
  const auto lanes_bits = [&](int v) {
    int b = 0;
    while (b < 6 && (1 << b) * v < a.fh) ++b;
    return b;
  };
  const auto fits = [&](int v) {
    return a.fh % v == 0 && reinterpret_cast<uintptr_t>(a.vin) % (v * sizeof(T)) == 0 &&
           reinterpret_cast<uintptr_t>(a.g) % (v * sizeof(float)) == 0;
  };
  int v = 4;
  while (v > 1 && (!fits(v) || (a.fh <= HC_WAVE * (v / 2) && ((int64_t)a.H << lanes_bits(v / 2)) <= HC_WAVE))) v /= 2;
  a.lph_bits = lanes_bits(v);
  const int64_t blocks = ((a.E + HC_WAVE - 1) / HC_WAVE + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
  if (!hc_grid_ok(blocks)) return HC_EUNSUPPORTED;
  const dim3 grid((unsigned)blocks), block(HC_BLOCK);
  if (v == 4) edge_grad_rows<T, 4, 8><<<grid, block, 0, st>>>(a);
  else if (v == 2) edge_grad_rows<T, 2, 8><<<grid, block, 0, st>>>(a);
  else edge_grad_rows<T, 1, 16><<<grid, block, 0, st>>>(a);
  return hc_launch_status();
}

}  // namespace

int hc_edge_grad(const int64_t *ptr, const int64_t *idx, const float *g, const int64_t *hmap, const void *vin, int in_dtype,
                 float *edge_grad, int64_t E, int64_t R, int64_t F, int64_t n_head, hipStream_t st) {
  if (E <= 0) return HC_OK;
  EdgeGradArgs a{ptr, idx, g, hmap, vin, edge_grad, E, R, (int)n_head, (int)F, 0};
  if (in_dtype == HC_F32) return eg_launch<float>(a, st);
  if (in_dtype == HC_F16) return eg_launch<__half>(a, st);
  return eg_launch<__hip_bfloat16>(a, st);
}
