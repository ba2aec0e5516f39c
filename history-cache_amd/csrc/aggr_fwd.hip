// hc_aggr_fwd: argument checks, the long rows' lists, and the choice of the kernel (aggr_fwd_rows.h; one
// translation unit per element type, aggr_fwd_f32.hip / _f16.hip / _bf16.hip).
#include "aggr_fwd_rows.h"

namespace {

// Notes the long rows of a tile in the lists.
__global__ __launch_bounds__(HC_BLOCK) void fwd_find_long(FwdArgs a) {
  __shared__ int n_near, n_far, n_staged;
  if (threadIdx.x == 0) n_near = n_far = n_staged = 0;
  __syncthreads();
  const int64_t total = a.ptr[a.R] - a.ptr[0];
  const int64_t far_above = fwd_far_above(a, total);
  const int64_t first = (int64_t)blockIdx.x * a.tile;
  const int64_t last = first + a.tile < a.R ? first + a.tile : a.R;
  const int64_t staged_above = a.stage != nullptr ? fwd_staged_above(a, total) : INT64_MAX;
  const int64_t staged0 = a.stage != nullptr ? seg_part(a.ptr, first, staged_above) : 0;
  const int64_t near0 = seg_part(a.ptr, first, a.slice_above), far0 = seg_part(a.ptr, first, far_above);
  constexpr int ITEMS = 4;
  for (int64_t r0 = first; r0 < last; r0 += HC_BLOCK * ITEMS) {
    int64_t deg[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int64_t r = r0 + it * HC_BLOCK + threadIdx.x;
      deg[it] = r < last ? a.ptr[r + 1] - a.ptr[r] : 0;
    }
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int64_t r = r0 + it * HC_BLOCK + threadIdx.x;
      if (deg[it] <= a.slice_above || (a.hmap != nullptr && a.hmap[r] != -1)) continue;
      if (deg[it] > staged_above) {
        const int64_t p = staged0 + atomicAdd(&n_staged, 1);
        if (p < a.staged.cap) a.staged.item[p] = (int32_t)r;
      } else if (deg[it] > far_above) {
        const int64_t p = far0 + atomicAdd(&n_far, 1);
        if (p < a.far.cap) a.far.item[p] = (int32_t)r;
      } else {
        const int64_t p = near0 + atomicAdd(&n_near, 1);
        if (p < a.near.cap) a.near.item[p] = (int32_t)r;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (blockIdx.x == 0) {
      a.plan->far_above = far_above;
      a.plan->staged_above = staged_above;
      a.plan->listed = total / (far_above + 1) <= a.far.cap &&
                       (a.split_above == 0 || total / (a.slice_above + 1) <= a.near.cap) ? 1 : 0;
    }
    a.near.count[blockIdx.x] = n_near;
    a.far.count[blockIdx.x] = n_far;
    if (a.stage != nullptr) a.staged.count[blockIdx.x] = n_staged;
  }
}

// Source tables below this size go without the one-bit-per-source filter in front of the map lookup:
// their map (8 bytes per source) stays in the L2s anyway.
constexpr int64_t FWD_BITS_MIN_SRC = (int64_t)1 << 20;
constexpr int64_t FWD_SELF_EDGES = 65536;       // at most FWD_SELF_ITEMS rows above FWD_HEAD_SLICE_EDGES
constexpr int FWD_FRONT_BLOCKS = 2048;
constexpr int FWD_SELF_FRONT_BLOCKS = 128;

struct FwdScratch {
  void *ptr;
  size_t bytes;
};

// Workspace of a forward launch: the two lists (their counts and the plan, then their entries: a third of the room for
// whole rows, two thirds for sliced ones), then one bit per source (per-source substitution over many
// sources).  Either part may be absent (0 bytes).
constexpr size_t FWD_COUNT_BYTES = 2 * SEG_MAX_REGIONS * sizeof(int32_t);
constexpr size_t FWD_HEAD_BYTES = FWD_COUNT_BYTES + 256;
// For rows of several heads, 4 adjacent columns of a row in one head: the list of the rows to be staged and the room for their
// copies, in front of the other lists.  Blocks of fewer edges are not worth the launch that copies (3 us where there is
// nothing to copy); a copy of all edges is not needed, and copies of more than 96 MB would be bound by the memory
// like the launch itself.
constexpr int64_t FWD_STAGE_MIN_EDGES = (int64_t)1 << 18;
constexpr int64_t FWD_STAGE_BYTES = (int64_t)96 << 20;
constexpr size_t FWD_STAGE_LIST_BYTES = (SEG_MAX_REGIONS + 3 * FWD_STAGED_ROWS + 64) * sizeof(int32_t);    // counts, list, order
size_t fwd_stage_bytes(int mode, int64_t E, int64_t F, int64_t n_head) {
  if (mode != HC_SUBST_ROW || n_head <= 1 || F % FWD_STAGED_COLS != 0 || E < FWD_STAGE_MIN_EDGES || F > 0x3fffffffLL / n_head) return 0;
  const int64_t edge = (F + 1) * n_head * (int64_t)sizeof(float);
  const int64_t most = E + FWD_STAGED_ROWS * FWD_STAGED_UNIT;      // every row's copy is a whole number of units
  return FWD_STAGE_LIST_BYTES + (size_t)(most < FWD_STAGE_BYTES / edge ? hc_align_up((size_t)(most * edge), 256) : FWD_STAGE_BYTES);
}

struct FwdWsLayout {
  size_t list_bytes, bits_bytes, total;
};
FwdWsLayout fwd_ws_layout(int mode, int64_t R, int64_t E, int64_t n_src) {
  FwdWsLayout L{0, 0, 0};
  if (E > FWD_HEAD_SLICE_EDGES && !(R <= FWD_SELF_ROWS && E <= FWD_SELF_EDGES)) {
    const int64_t near = E / (HC_LONG_ROW_EDGES + 1) + 1;
    L.list_bytes = hc_align_up(FWD_HEAD_BYTES + (size_t)(3 * near + 3) * sizeof(int32_t), 256);
  }
  if (mode == HC_SUBST_SRC && n_src >= FWD_BITS_MIN_SRC) L.bits_bytes = hc_align_up((size_t)((n_src + 63) / 64) * 8, 256);
  L.total = L.list_bytes + L.bits_bytes;
  return L;
}

// bits[s] = (hmap[s] != -1), 64 sources per ballot.  The map is read with ordinary loads: this pass also
// brings it into the last-level cache in front of the launch that looks sources up in it.
__global__ __launch_bounds__(HC_BLOCK) void fwd_src_bits(const int64_t *__restrict__ hmap, int64_t n_src,
                                                          unsigned long long *__restrict__ bits) {
  const int lane = hc_lane();
  const int64_t stride = (int64_t)gridDim.x * HC_WAVES_PER_BLOCK * HC_WAVE;
  for (int64_t base = ((int64_t)blockIdx.x * HC_WAVES_PER_BLOCK + hc_wave_in_block()) * HC_WAVE; base < n_src;
       base += stride) {
    const bool has = base + lane < n_src && hmap[base + lane] != -1;
    const unsigned long long b = __ballot(has);
    if (lane == 0) bits[base / HC_WAVE] = b;
  }
}

// The lists' launch and the front blocks of the main one.  `max_degree` >= 0: no row has more edges.
int fwd_prepare_lists(FwdArgs &a, bool src_mode, FwdScratch ws, int64_t n_src, int64_t max_degree, size_t stage_bytes,
                      hipStream_t st) {
  const bool ws_ok = ws.ptr != nullptr && reinterpret_cast<uintptr_t>(ws.ptr) % 256 == 0;
  if (ws_ok && stage_bytes > 0 && ws.bytes > stage_bytes + FWD_HEAD_BYTES && max_degree < 0 && a.R <= 0x7fffffffLL) {
    a.staged.count = static_cast<int32_t *>(ws.ptr);
    a.staged.item = a.staged.count + SEG_MAX_REGIONS;
    a.staged.cap = FWD_STAGED_ROWS;
    a.staged_order = a.staged.item + FWD_STAGED_ROWS;
    a.stage = reinterpret_cast<float *>(static_cast<char *>(ws.ptr) + FWD_STAGE_LIST_BYTES);
    a.stage_floats = (int64_t)((stage_bytes - FWD_STAGE_LIST_BYTES) / sizeof(float));
    ws.ptr = static_cast<char *>(ws.ptr) + stage_bytes;
    ws.bytes -= stage_bytes;
  }
  // the caller sized the workspace with hc_aggr_fwd_workspace_bytes(mode, R, E, n_src): the bitmap, when
  // there is one, takes the last bits_bytes bytes and the lists what lies in front of it
  size_t room = ws_ok ? ws.bytes : 0;
  if (ws_ok && src_mode && n_src >= FWD_BITS_MIN_SRC) {
    const size_t bb = hc_align_up((size_t)((n_src + 63) / 64) * 8, 256);
    if (ws.bytes >= bb) {
      room = (ws.bytes - bb) / 256 * 256;
      unsigned long long *bits = reinterpret_cast<unsigned long long *>(static_cast<char *>(ws.ptr) + room);
      fwd_src_bits<<<dim3(2048), dim3(HC_BLOCK), 0, st>>>(a.hmap, n_src, bits);
      a.src_bits = reinterpret_cast<const uint32_t *>(bits);
    }
  }
  if (max_degree >= 0 && max_degree <= a.slice_above) {
    a.split_above = a.slice_above = 0;
    return HC_OK;
  }
  if (a.R > 0x7fffffffLL) return HC_OK;
  if (room > FWD_HEAD_BYTES + 3 * sizeof(int32_t)) {
    a.tile = seg_tile(a.R);
    a.n_tiles = (int)((a.R + a.tile - 1) / a.tile);
    const int64_t items = (int64_t)((room - FWD_HEAD_BYTES) / sizeof(int32_t));
    a.near.count = static_cast<int32_t *>(ws.ptr);
    a.far.count = a.near.count + SEG_MAX_REGIONS;
    a.plan = reinterpret_cast<FwdPlan *>(static_cast<char *>(ws.ptr) + FWD_COUNT_BYTES);
    a.near.item = reinterpret_cast<int32_t *>(static_cast<char *>(ws.ptr) + FWD_HEAD_BYTES);
    a.near.cap = items / 3;
    a.far.item = a.near.item + a.near.cap;
    a.far.cap = items - a.near.cap;
    const int64_t blocks = (items + 3) / 4;      // a generous share even when every entry is one task
    a.front = (int)(blocks < 64 ? 64 : (blocks > FWD_FRONT_BLOCKS ? FWD_FRONT_BLOCKS : blocks));
    FwdArgs f = a;
    if (src_mode) f.hmap = nullptr;
    fwd_find_long<<<dim3((unsigned)a.n_tiles), dim3(HC_BLOCK), 0, st>>>(f);
  } else if (a.R <= FWD_SELF_ROWS) {
    a.front = FWD_SELF_FRONT_BLOCKS;
  }
  if (a.n_tiles == 0) a.stage = nullptr;       // no room for the lists behind the copies
  return HC_OK;
}

}  // namespace

extern "C" int64_t hc_aggr_fwd_long_row_edges(int64_t F, int in_dtype) {
  if (in_dtype < HC_F32 || in_dtype > HC_BF16 || F <= 0) return 0;
  return HC_LONG_ROW_EDGES;
}

extern "C" size_t hc_aggr_fwd_workspace_bytes(int mode, int64_t R, int64_t E, int64_t n_src) {
  if (R < 0 || E < 0 || n_src < 0) return 0;
  return fwd_ws_layout(mode, R, E, n_src).total;
}

extern "C" int hc_aggr_fwd(int mode, const int64_t *ptr, const int64_t *idx, const void *vin,
                           int in_dtype, const int64_t *hmap, const void *hbuf, int hist_dtype,
                           int64_t hsize, const float *edge_value, int64_t n_head, float *vout,
                           int64_t R, int64_t F, int64_t n_src, void *workspace,
                           size_t workspace_bytes, void *stream) {
  return hc_aggr_fwd_bounded(mode, ptr, idx, vin, in_dtype, hmap, hbuf, hist_dtype, hsize, edge_value, n_head, vout,
                             R, F, n_src, -1, workspace, workspace_bytes, stream);
}

extern "C" int hc_aggr_fwd_bounded(int mode, const int64_t *ptr, const int64_t *idx, const void *vin,
                                   int in_dtype, const int64_t *hmap, const void *hbuf, int hist_dtype,
                                   int64_t hsize, const float *edge_value, int64_t n_head, float *vout,
                                   int64_t R, int64_t F, int64_t n_src, int64_t max_degree, void *workspace,
                                   size_t workspace_bytes, void *stream) {
  return hc_aggr_fwd_for(mode, ptr, idx, vin, in_dtype, hmap, hbuf, hist_dtype, hsize, edge_value, n_head, vout, R, F,
                         n_src, -1, max_degree, workspace, workspace_bytes, stream);
}

extern "C" size_t hc_aggr_fwd_workspace_bytes_for(int mode, int64_t R, int64_t E, int64_t n_src, int64_t F, int64_t n_head) {
  if (R < 0 || E < 0 || n_src < 0 || F < 1 || n_head < 1) return 0;
  const size_t lists = fwd_ws_layout(mode, R, E, n_src).total;
  return lists > 0 ? lists + fwd_stage_bytes(mode, E, F, n_head) : 0;
}

extern "C" int hc_aggr_fwd_for(int mode, const int64_t *ptr, const int64_t *idx, const void *vin, int in_dtype,
                               const int64_t *hmap, const void *hbuf, int hist_dtype, int64_t hsize,
                               const float *edge_value, int64_t n_head, float *vout, int64_t R, int64_t F, int64_t n_src,
                               int64_t E, int64_t max_degree, void *workspace, size_t workspace_bytes, void *stream) {
  const FwdScratch ws{workspace, workspace ? workspace_bytes : 0};
  HC_REQUIRE(R >= 0 && F > 0 && n_src >= 0 && n_head >= 1);
  if (R == 0) return HC_OK;
  HC_REQUIRE(ptr && vout);
  HC_REQUIRE(mode == HC_SUBST_ROW || mode == HC_SUBST_SRC);
  if (in_dtype < HC_F32 || in_dtype > HC_BF16) return HC_EDTYPE;
  if (hmap && (hist_dtype < HC_F32 || hist_dtype > HC_BF16)) return HC_EDTYPE;
  if (hmap) HC_REQUIRE(hbuf != nullptr && hsize > 0);
  if (n_head > 1) HC_REQUIRE(edge_value != nullptr);
  const int src_mode = (mode == HC_SUBST_SRC) ? 1 : 0;
  if (src_mode) {
    if (edge_value) return HC_EUNSUPPORTED;
    if (hmap) {
      HC_REQUIRE(hsize >= F);
      // the table has the features' element type, or the features are fp32 and the table is narrower
      if (hist_dtype != in_dtype && in_dtype != HC_F32) return HC_EUNSUPPORTED;
    }
  } else if (hmap) {
    HC_REQUIRE(hsize == F * n_head || (hsize >= F && n_head == 1) || hsize == F);
  }
  if (n_head > 0x7fffffffLL || F > 0x3fffffffLL / n_head) return HC_EUNSUPPORTED;
  FwdArgs a{};
  a.ptr = ptr;
  a.idx = idx;
  a.vin = vin;
  a.hmap = hmap;
  a.hbuf = hbuf;
  a.hist_dtype = hmap ? hist_dtype : in_dtype;
  a.hsize = hsize;
  a.ev = edge_value;
  a.n_head = (int)n_head;
  a.vout = vout;
  a.R = R;
  a.F = F * n_head;                 // a row is all heads side by side
  a.small_matrix = n_src <= (int64_t)(0xffffffffull / ((size_t)a.F * (in_dtype == HC_F32 ? 4 : 2)));
  a.split_above = n_head > 1 ? 0 : HC_LONG_ROW_EDGES;
  a.slice_above = n_head > 1 ? FWD_HEAD_SLICE_EDGES : HC_LONG_ROW_EDGES;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int rc = fwd_prepare_lists(a, src_mode != 0 && hmap != nullptr, ws, n_src, max_degree,
                                   fwd_stage_bytes(mode, E, F, n_head), st);
  if (rc != HC_OK) return rc;
  if (in_dtype == HC_F32) return fwd_dispatch_f32(a, src_mode != 0, (int)n_head, st);
  if (in_dtype == HC_F16) return fwd_dispatch_f16(a, src_mode != 0, (int)n_head, st);
  return fwd_dispatch_bf16(a, src_mode != 0, (int)n_head, st);
}
