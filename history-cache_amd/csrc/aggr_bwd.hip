// hc_aggr_bwd: argument checks, the long sources' lists and the runs of sources, the choice of the kernel
// (aggr_bwd_rows.h; one translation unit per element type of the gradient, aggr_bwd_f32.hip / _f16.hip /
// _bf16.hip); the gradient of the history buffer of several heads; the relational layer's backward.
#include "aggr_bwd_rows.h"

namespace {

// Notes the long sources of a tile in the two lists and where the runs that start in it begin.  One thread per
// source; source n_src stands for the end.
constexpr int BWD_PREP_BLOCK = 1024;     // at most SEG_MAX_REGIONS blocks: large ones, to fill the chip
__global__ __launch_bounds__(BWD_PREP_BLOCK) void bwd_prepare(BwdArgs a, int64_t runs) {
  __shared__ int n_mid, n_hub, n_giant;
  if (threadIdx.x == 0) n_mid = n_hub = n_giant = 0;
  for (int64_t i = (int64_t)blockIdx.x * BWD_PREP_BLOCK + threadIdx.x; i < a.n_tickets; i += (int64_t)gridDim.x * BWD_PREP_BLOCK)
    a.ticket[i] = 0u;
  __syncthreads();
  const int64_t first = (int64_t)blockIdx.x * a.tile;
  int64_t last = first + a.tile;
  if (last > a.n_src) last = a.n_src;
  const bool at_end = last == a.n_src;
  const int64_t mid0 = seg_part(a.ptrT, first, a.long_above);
  const int64_t hub0 = a.chunk > 0 ? seg_part(a.ptrT, first, a.chunk) : 0;
  const int64_t giant0 = a.giant.cap > 0 ? seg_part(a.ptrT, first, BWD_SPAN) : 0;
  constexpr int ITEMS = 4;
  for (int64_t s0 = first; s0 < last + (at_end ? 1 : 0); s0 += BWD_PREP_BLOCK * ITEMS) {
    int64_t p[ITEMS], p1[ITEMS], pm[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int64_t s = s0 + it * BWD_PREP_BLOCK + threadIdx.x;
      const bool in = s < last || (at_end && s == last);
      p[it] = in ? a.ptrT[s] : -1;
      p1[it] = s < last ? a.ptrT[s + 1] : p[it];
      pm[it] = in && s > 0 ? a.ptrT[s - 1] : 0;
    }
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      if (p[it] < 0) continue;
      const int64_t s = s0 + it * BWD_PREP_BLOCK + threadIdx.x;
      if (a.run_start_out != nullptr) {
        int64_t hi = (p[it] + (int64_t)BWD_SRC_COST * s) / BWD_UNIT;
        if (hi >= runs) hi = runs - 1;
        int64_t lo = s > 0 ? (pm[it] + (int64_t)BWD_SRC_COST * (s - 1)) / BWD_UNIT + 1 : 0;
        for (; lo <= hi; ++lo) a.run_start_out[lo] = (int32_t)s;
      }
      const int64_t deg = p1[it] - p[it];
      if (deg <= a.long_above) continue;
      if (a.giant.cap > 0 && deg > BWD_SPAN) {
        const int64_t at = giant0 + atomicAdd(&n_giant, 1);
        if (at < a.giant.cap) a.giant.item[at] = (int32_t)s;
      } else if (a.chunk > 0 && deg > a.chunk) {
        const int64_t at = hub0 + atomicAdd(&n_hub, 1);
        if (at < a.hub.cap) a.hub.item[at] = (int32_t)s;
      } else {
        const int64_t at = mid0 + atomicAdd(&n_mid, 1);
        if (at < a.mid.cap) a.mid.item[at] = (int32_t)s;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const bool fits = a.ptrT[a.n_src] - a.ptrT[0] <= a.E;      // else the lists may lack entries: none is used
    a.mid.count[blockIdx.x] = fits ? n_mid : 0;
    a.hub.count[blockIdx.x] = fits ? n_hub : 0;
    a.giant.count[blockIdx.x] = fits ? n_giant : 0;
  }
}

bool bwd_fast_shape(int64_t F) {
  return F == 64 || F == 128 || F == 192 || F == 256 || F == 384 || F == 512 || F == 768 || F == 1024;
}

// Workspace: the lists' counts and entries, the giants' tickets and chunk sums (F: the width of a chunked sum, else 0),
// then the runs' starts.  A block of up to BWD_LONG edges has no long source and needs none of them.
struct BwdWsLayout {
  size_t mid, hub, giant, ticket, partial, lists, run_start, total;
  int64_t mid_cap, hub_cap, giant_cap, tickets, runs;
};
BwdWsLayout bwd_ws_layout(int64_t E, int64_t F, int64_t n_src) {
  BwdWsLayout L{};
  if (E <= BWD_LONG) return L;
  L.mid_cap = E / (BWD_LONG + 1) + 1;
  L.hub_cap = E / (BWD_CHUNK + 1) + 1;
  L.giant_cap = F > 0 && E > BWD_SPAN ? E / (BWD_SPAN + 1) + 1 : 0;
  L.tickets = L.giant_cap * ((F + BWD_SLICE - 1) / BWD_SLICE);
  L.mid = 3 * SEG_MAX_REGIONS * sizeof(int32_t);
  L.hub = L.mid + (size_t)L.mid_cap * sizeof(int32_t);
  L.giant = L.hub + (size_t)L.hub_cap * sizeof(int32_t);
  L.ticket = L.giant + (size_t)L.giant_cap * sizeof(int32_t);
  L.partial = hc_align_up(L.ticket + (size_t)L.tickets * sizeof(int32_t), 256);
  L.lists = L.partial;
  if (L.giant_cap > 0) L.lists += hc_align_up((size_t)(2 * (E / BWD_CHUNK + 1)) * (size_t)F * sizeof(float), 256);
  L.run_start = L.lists;
  L.runs = (E + BWD_SRC_COST * n_src) / BWD_UNIT + 1;
  L.total = L.lists + hc_align_up((size_t)L.runs * sizeof(int32_t), 256);
  return L;
}

// grad_hbuf[R, hsize] of several heads (heads summed when hsize == F, concatenated when
// hsize == F*H; columns beyond the written span are 0).
__global__ __launch_bounds__(HC_BLOCK) void bwd_hist_generic(const float *__restrict__ g,
                                                              const int64_t *__restrict__ hmap,
                                                              float *__restrict__ grad_hbuf,
                                                              int64_t hsize, int64_t R, int64_t F,
                                                              int64_t H) {
  const int lane = hc_lane();
  const int64_t row = (int64_t)blockIdx.x * HC_WAVES_PER_BLOCK + hc_wave_in_block();
  if (row >= R) return;
  const bool hit = hmap[row] != -1;
  float *__restrict__ d = grad_hbuf + row * hsize;
  const float *__restrict__ s = g + row * H * F;
  const bool concat = (H > 1 && hsize == F * H);
  for (int64_t c = lane; c < hsize; c += HC_WAVE) {
    float v = 0.0f;
    if (hit) {
      if (concat) {
        v = s[c];
      } else if (c < F) {
        for (int64_t h = 0; h < H; ++h) v += s[h * F + c];
      }
    }
    d[c] = v;
  }
}

// The sums of the sources (and grad_hbuf of a single head).  `vin_dtype` is grad_vin's element type.
int bwd_sum_sources(BwdArgs &a, int64_t E, void *workspace, size_t workspace_bytes, int vin_dtype, bool masked,
                    hipStream_t st) {
  a.hist_blocks = (a.grad_hbuf && a.n_head == 1) ? (a.R + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK : 0;
  const bool chunked = a.ev == nullptr && bwd_fast_shape(a.F);
  const BwdWsLayout L = bwd_ws_layout(E, chunked ? a.F : 0, a.n_src);
  char *ws = static_cast<char *>(workspace);
  // fixed runs: enough of them for the chip, at most BWD_MAX_RUN sources (two layers of a sampled batch: 31 us, in
  // runs of 32 whatever their number 40 us)
  a.run = (int)(a.n_src / 4096);
  a.run = a.run < 4 ? 4 : (a.run > BWD_MAX_RUN ? BWD_MAX_RUN : a.run);
  int64_t waves = (a.n_src + a.run - 1) / a.run;
  // (without rows every edge of a shared view is stepped over: nothing to share out, and no row of g to read instead)
  if (L.lists > 0 && a.n_src > 0 && a.R > 0 && ws != nullptr && workspace_bytes >= L.lists && reinterpret_cast<uintptr_t>(ws) % 256 == 0) {
    a.E = E;
    a.long_above = BWD_LONG;
    a.chunk = chunked ? BWD_CHUNK : 0;
    a.tile = seg_tile(a.n_src);
    a.n_tiles = (int)((a.n_src + a.tile - 1) / a.tile);
    a.mid.count = reinterpret_cast<int32_t *>(ws);
    a.hub.count = a.mid.count + SEG_MAX_REGIONS;
    a.giant.count = a.hub.count + SEG_MAX_REGIONS;
    a.giant.item = reinterpret_cast<int32_t *>(ws + L.giant);
    a.giant.cap = L.giant_cap;
    a.ticket = reinterpret_cast<uint32_t *>(ws + L.ticket);
    a.n_tickets = L.tickets;
    a.partial = reinterpret_cast<float *>(ws + L.partial);
    a.mid.item = reinterpret_cast<int32_t *>(ws + L.mid);
    a.hub.item = reinterpret_cast<int32_t *>(ws + L.hub);
    a.mid.cap = L.mid_cap;
    a.hub.cap = L.hub_cap;
    int64_t runs = 0;
    if (workspace_bytes >= L.total) {
      a.run_start_out = reinterpret_cast<int32_t *>(ws + L.run_start);
      a.run_start = a.run_start_out;
      waves = runs = L.runs;
    }
    const int64_t tasks = (L.mid_cap * ((a.F + BWD_SLICE - 1) / BWD_SLICE) + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
    a.front = (int)(tasks < 64 ? 64 : (tasks > BWD_FRONT_BLOCKS ? BWD_FRONT_BLOCKS : tasks));
    bwd_prepare<<<dim3((unsigned)a.n_tiles), dim3(BWD_PREP_BLOCK), 0, st>>>(a, runs);
    if (hc_launch_status() != HC_OK) return HC_ELAUNCH;
  }
  a.src_blocks = (waves + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
  if (a.src_blocks + a.hist_blocks == 0) return HC_OK;
  if (vin_dtype == HC_F32) return bwd_dispatch_f32(a, masked, st);
  if (vin_dtype == HC_F16) return bwd_dispatch_f16(a, masked, st);
  return bwd_dispatch_bf16(a, masked, st);
}

// ---------------------------------------------------------------------------------------
// Relational layer over the mini-batch's shared view.  The layer's forward sums, for every (row, relation)
// group, x[src] * (1 / deg(row)) over the group's kept edges; here source s collects
// g[row * K + rel(e), :] * (1 / deg(row)) over its kept edges in ascending (row, edge slot) order: the order
// of the batch view, so that no view of the regrouped block has to be built.  An edge is kept under
// hc_typed_csr's rule: row < R, slot < E, relation in [0, K), source flagged in `used` (when given).
// One wave per source; up to UNROLL gradient rows in flight; products rounded, then added in order.
// ---------------------------------------------------------------------------------------
template <int VEC, int CHUNKS, int UNROLL>
__global__ __launch_bounds__(HC_BLOCK) void bwd_typed_batch_view(
    const int64_t *__restrict__ ptr, const int64_t *__restrict__ ptrT, const int32_t *__restrict__ rowT,
    const int32_t *__restrict__ edgeT, const int64_t *__restrict__ et, const uint8_t *__restrict__ used,
    const float *__restrict__ g, float *__restrict__ grad_vin, int64_t R, int64_t E, int K, int64_t n_src) {
  constexpr int F = HC_WAVE * VEC * CHUNKS;
  const int lane = hc_lane();
  const int64_t s = (int64_t)blockIdx.x * HC_WAVES_PER_BLOCK + hc_wave_in_block();
  if (s >= n_src) return;
  float acc[CHUNKS][VEC];
#pragma unroll
  for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
    for (int i = 0; i < VEC; ++i) acc[k][i] = 0.0f;
  const bool src_kept = used == nullptr || used[s] != 0;
  const int64_t begin = src_kept ? ptrT[s] : 0;
  const int64_t end = src_kept ? ptrT[s + 1] : 0;
  for (int64_t base = begin; base < end; base += HC_WAVE) {
    const int64_t left = end - base;
    const int n = left < HC_WAVE ? (int)left : HC_WAVE;
    int64_t my_group = -1;
    float my_w = 0.0f;
    if (lane < n) {
      const int64_t row = rowT[base + lane];
      const int64_t e = edgeT[base + lane];
      if (row < R && e < E) {
        const int64_t rel = et[e];
        const int64_t d = ptr[row + 1] - ptr[row];      // 0: a row that the layer's own offsets leave empty
        if (rel >= 0 && rel < K && d > 0) {
          my_group = row * K + rel;
          my_w = 1.0f / (float)d;
        }
      }
    }
    unsigned long long todo = __ballot(my_group >= 0);
    while (todo != 0ull) {
      float v[UNROLL][CHUNKS][VEC];
      float w[UNROLL];
      bool on[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        w[u] = 0.0f;
        on[u] = todo != 0ull;
        if (on[u]) {
          const int j = __builtin_ctzll(todo);
          todo &= todo - 1ull;
          w[u] = hc_readlane_f(my_w, j);
          const float *p = g + hc_readlane64(my_group, j) * F + lane * VEC;
#pragma unroll
          for (int k = 0; k < CHUNKS; ++k) hc_vec<float, VEC>::load(p + k * HC_WAVE * VEC, v[u][k]);
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        if (on[u]) {
#pragma unroll
          for (int k = 0; k < CHUNKS; ++k)
#pragma unroll
            for (int i = 0; i < VEC; ++i) acc[k][i] += __fmul_rn(v[u][k][i], w[u]);
        }
      }
    }
  }
  float *__restrict__ o = grad_vin + s * F + lane * VEC;
#pragma unroll
  for (int k = 0; k < CHUNKS; ++k) hc_vec<float, VEC>::store(o + k * HC_WAVE * VEC, acc[k]);
}

}  // namespace

extern "C" size_t hc_aggr_bwd_workspace_bytes(int64_t E_total, int64_t F) {
  if (E_total < 0 || F <= 0) return 0;
  return bwd_ws_layout(E_total, bwd_fast_shape(F) ? F : 0, 0).lists;
}

extern "C" size_t hc_aggr_bwd_workspace_bytes_for(int64_t E_total, int64_t F, int64_t n_src) {
  if (E_total < 0 || F <= 0 || n_src < 0) return 0;
  return bwd_ws_layout(E_total, bwd_fast_shape(F) ? F : 0, n_src).total;
}

extern "C" int64_t hc_aggr_bwd_chunk_edges(int64_t F) { return bwd_fast_shape(F) ? BWD_CHUNK : 0; }

namespace {

int aggr_bwd_impl(const int64_t *ptr, const int64_t *idx, const int64_t *ptrT,
                  const int32_t *rowT, const int32_t *edgeT, const float *g,
                  const int64_t *hmap, const float *edge_value, const void *vin, int in_dtype,
                  int64_t n_head, void *grad_vin, int vin_dtype, float *grad_hbuf, int64_t hsize,
                  float *edge_grad, int64_t E_total, int64_t R, int64_t F, int64_t n_src,
                  void *workspace, size_t workspace_bytes, bool masked, void *stream) {
  HC_REQUIRE(R >= 0 && F > 0 && n_src >= 0 && n_head >= 1 && E_total >= 0);
  HC_REQUIRE(ptr && ptrT);
  HC_REQUIRE(g || R == 0);   // a layer without rows has no gradient rows to read
  HC_REQUIRE(grad_vin || n_src == 0);
  if (vin_dtype < HC_F32 || vin_dtype > HC_BF16) return HC_EDTYPE;
  if (n_head > 1) HC_REQUIRE(edge_value != nullptr);
  if (grad_hbuf) HC_REQUIRE(hmap != nullptr && hsize >= F);
  if (grad_hbuf && n_head > 1) HC_REQUIRE(hsize == F || hsize == F * n_head);
  if (edge_grad) {
    HC_REQUIRE(edge_value && vin && idx);
    if (in_dtype < HC_F32 || in_dtype > HC_BF16) return HC_EDTYPE;
  }
  if (edge_value) HC_REQUIRE(edgeT != nullptr);
  HC_REQUIRE(rowT != nullptr || n_src == 0);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int64_t lim = 0x7ffffffeLL;
  if (R > lim) return HC_EUNSUPPORTED;

  if (n_head > 0x7fffffffLL || F > 0x3fffffffLL / n_head) return HC_EUNSUPPORTED;
  BwdArgs a{};
  a.ptr = ptr;
  a.ptrT = ptrT;
  a.rowT = rowT;
  a.edgeT = edgeT;
  a.ev = edge_value;
  a.n_head = (int)n_head;
  a.g = g;
  a.hmap = hmap;
  a.grad_vin = grad_vin;
  a.grad_hbuf = grad_hbuf;
  a.hsize = hsize;
  a.R = R;
  a.n_src = n_src;
  a.F = F * n_head;
  a.small_matrix = R <= (int64_t)(0xffffffffull / ((size_t)a.F * sizeof(float)));
  const int rc = bwd_sum_sources(a, E_total, workspace, workspace_bytes, vin_dtype, masked, st);
  if (rc != HC_OK) return rc;
  if (grad_hbuf && n_head > 1 && R > 0) {
    const int64_t hb = (R + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
    if (!hc_grid_ok(hb)) return HC_EUNSUPPORTED;
    bwd_hist_generic<<<dim3((unsigned)hb), dim3(HC_BLOCK), 0, st>>>(g, hmap, grad_hbuf, hsize, R, F, n_head);
    if (hc_launch_status() != HC_OK) return HC_ELAUNCH;
  }
  if (edge_grad) return hc_edge_grad(ptr, idx, g, hmap, vin, in_dtype, edge_grad, E_total, R, F, n_head, st);
  return HC_OK;
}

}  // namespace

extern "C" int hc_aggr_bwd(const int64_t *ptr, const int64_t *idx, const int64_t *ptrT,
                           const int32_t *rowT, const int32_t *edgeT, const float *g,
                           const int64_t *hmap, const float *edge_value, const void *vin, int in_dtype,
                           int64_t n_head, float *grad_vin, float *grad_hbuf, int64_t hsize,
                           float *edge_grad, int64_t E_total, int64_t R, int64_t F, int64_t n_src,
                           void *workspace, size_t workspace_bytes, void *stream) {
  return aggr_bwd_impl(ptr, idx, ptrT, rowT, edgeT, g, hmap, edge_value, vin, in_dtype, n_head, grad_vin, HC_F32,
                       grad_hbuf, hsize, edge_grad, E_total, R, F, n_src, workspace, workspace_bytes, false,
                       stream);
}

extern "C" int hc_aggr_bwd_as(const int64_t *ptr, const int64_t *idx, const int64_t *ptrT,
                              const int32_t *rowT, const int32_t *edgeT, const float *g,
                              const int64_t *hmap, const float *edge_value, const void *vin, int in_dtype,
                              int64_t n_head, void *grad_vin, int grad_dtype, float *grad_hbuf, int64_t hsize,
                              float *edge_grad, int64_t E_total, int64_t R, int64_t F, int64_t n_src,
                              void *workspace, size_t workspace_bytes, void *stream) {
  return aggr_bwd_impl(ptr, idx, ptrT, rowT, edgeT, g, hmap, edge_value, vin, in_dtype, n_head, grad_vin, grad_dtype,
                       grad_hbuf, hsize, edge_grad, E_total, R, F, n_src, workspace, workspace_bytes, false,
                       stream);
}

extern "C" int hc_aggr_bwd_batch_view(const int64_t *ptr, const int64_t *ptrT, const int32_t *rowT,
                                      const float *g, const int64_t *hmap, float *grad_vin,
                                      float *grad_hbuf, int64_t hsize, int64_t E_view, int64_t R, int64_t F,
                                      int64_t n_src, void *workspace, size_t workspace_bytes, void *stream) {
  return hc_aggr_bwd_batch_view_as(ptr, ptrT, rowT, g, hmap, grad_vin, HC_F32, grad_hbuf, hsize, E_view, R, F, n_src,
                                   workspace, workspace_bytes, stream);
}

extern "C" int hc_aggr_bwd_batch_view_as(const int64_t *ptr, const int64_t *ptrT, const int32_t *rowT,
                                         const float *g, const int64_t *hmap, void *grad_vin, int grad_dtype,
                                         float *grad_hbuf, int64_t hsize, int64_t E_view, int64_t R, int64_t F,
                                         int64_t n_src, void *workspace, size_t workspace_bytes, void *stream) {
  return aggr_bwd_impl(ptr, nullptr, ptrT, rowT, nullptr, g, hmap, nullptr, nullptr, 0, 1, grad_vin, grad_dtype,
                       grad_hbuf, hsize, nullptr, E_view, R, F, n_src, workspace, workspace_bytes, true, stream);
}

extern "C" int hc_aggr_bwd_batch_view_typed(const int64_t *ptr, const int64_t *ptrT, const int32_t *rowT,
                                            const int32_t *edgeT, const int64_t *edge_types, int64_t E,
                                            int num_rel, const uint8_t *used_mask, const float *g,
                                            float *grad_vin, int64_t R, int64_t F, int64_t n_src, void *stream) {
  HC_REQUIRE(R >= 0 && F > 0 && n_src >= 0 && E >= 0 && num_rel >= 1);
  HC_REQUIRE(ptr && ptrT && g && edge_types);
  HC_REQUIRE(grad_vin || n_src == 0);
  HC_REQUIRE((rowT && edgeT) || n_src == 0);
  if (R > 0x7ffffffeLL / num_rel) return HC_EUNSUPPORTED;
  if (!bwd_fast_shape(F)) return HC_EUNSUPPORTED;
  if (reinterpret_cast<uintptr_t>(g) % 16 != 0 || reinterpret_cast<uintptr_t>(grad_vin) % 16 != 0)
    return HC_EUNSUPPORTED;
  if (n_src == 0) return HC_OK;
  const int64_t nb = (n_src + HC_WAVES_PER_BLOCK - 1) / HC_WAVES_PER_BLOCK;
  if (!hc_grid_ok(nb)) return HC_EUNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)nb), block(HC_BLOCK);
#define HC_TYPED(V, C)                                                                                  \
  if (F == 64 * (V) * (C))                                                                              \
    bwd_typed_batch_view<V, C, ((V) * (C) >= 16 ? 4 : 8)><<<grid, block, 0, st>>>(                      \
        ptr, ptrT, rowT, edgeT, edge_types, used_mask, g, grad_vin, R, E, num_rel, n_src);              \
  else
  HC_TYPED(4, 1) HC_TYPED(4, 2) HC_TYPED(4, 3) HC_TYPED(4, 4) HC_TYPED(2, 1) HC_TYPED(2, 3) HC_TYPED(1, 1)
  HC_TYPED(1, 3) return HC_EUNSUPPORTED;
#undef HC_TYPED
  return hc_launch_status();
}
