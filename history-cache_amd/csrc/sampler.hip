// Layered neighbour sampling on the device: produces the mini-batch wire format the model and the
// cache consume (/root/reference/hiscache/history_model.py:120-153, history_cache.py:307-324 read
// ptr / idx / sub_to_full / num_node_in_layer from the loader; the reference gets them from the
// external cxgnndl loader).  Sub-graph nodes are numbered seeds first, then every hop's new nodes in
// first-seen order; one shared CSR holds the sampled neighbours of all but the last hop's nodes.
//
// Per hop, for the frontier rows [lo, hi), four launches:
//   count    node map <- local ids of the frontier (the previous hop's new nodes); c(u) = min(deg(u), fanout),
//            summed up to every row inside its tile of 1024 rows, and per tile
//   pick     neighbour j of row u is position perm_u(j) of u's adjacency list (all of them, in
//            list order, when deg <= fanout); its full id goes to idx, and an integer atomicMin
//            leaves the first edge slot that mentions an unseen node in the node map
//   flag     an edge owns its node when the map holds its own slot: one bit per slot, the owners in front of every
//            64 slots inside their tile of 1024, and per tile
//   relabel  idx <- local ids (a new node's: the owners in front of its own, from the bits); owners append to
//            sub_to_full; the first thread writes the next hop's state (lo, hi, edges): every hop has a state of
//            its own, so nothing it reads changes under it
// The tiles' sums are added up by whoever needs the offset of a tile (hundreds of tiles: one or two loads per
// lane); beyond SP_DIRECT_TILES of them a launch of one block scans them first.  A batch is bound by its chain of
// small launches: with the library's scans (two launches each) and the commit of the new ids a hop took nine;
// a batch of 1000 seeds, fanouts 15, 10, 5, with its view 283 -> 246 us.
// perm_u is a keyed bijection of [0, deg): four Feistel rounds on the next even power of two with
// cycle walking, so the picks of a row are distinct (sampling without replacement) at O(fanout)
// work whatever the degree.  Everything is integer work with one well-defined result.
#include "hc_common.h"

namespace {

constexpr int32_t SP_UNSEEN = 0x7fffffff;
constexpr int32_t SP_PROV = 0x40000000;  // map values at or above this are edge slots, below are ids
// Lanes that share one row in the pick kernel: the fanout where two rows or more fit the wave so, else 16.  The kernel is
// bound by the arithmetic of the permutation (64-bit multiplications, walked until every lane of the wave is done), so
// what counts is how many lanes have a pick: three hops of 15, 10 and 5 from 1 000 seeds 55 us with groups of 16, now 42.
// Between 17 and 32 (three or two rows per wave instead of four that take two rounds each), groups of 16 / of the fanout, us:
// hops of 20 and 20 from 1 000 seeds, power-law degrees of 7 on average 55 / 49, of 15 64 / 55, every degree 100 84 / 76; from
// 20 000 seeds, power-law 7 101 / 93, every degree 7 (no row needs the permutation) 104 / 107; one hop of 25 or 32 from 20 000, power-law
// 15 46 / 42 and 45 / 43, every degree 7 35 / 35, 100 59 / 59 and 65 / 67.
constexpr int SP_GROUP = 16;
__host__ __device__ __forceinline__ int sp_group(int64_t fanout) { return fanout <= HC_WAVE / 2 ? (int)fanout : SP_GROUP; }
constexpr int SP_BLOCK = HC_BLOCK;       // threads of the kernels that own a tile
constexpr int SP_ITEMS = 4;
// Rows or edge slots per tile.  A hop has a hundred thousand of them: with tiles of 4096 (and blocks of 1024) a few
// tens of blocks stood in the chip, each behind its own chain of loads, and the three kernels took 86 us instead of 45.
constexpr int SP_TILE = SP_BLOCK * SP_ITEMS;
constexpr int64_t SP_DIRECT_TILES = 4096;

struct SpState {
  int64_t lo, hi;   // frontier rows of the current hop
  int64_t edges;    // edges written by earlier hops
  uint64_t key;     // the batch's sampling key
};

__host__ __device__ __forceinline__ uint64_t sp_mix64(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Keyed bijection of [0, d), d >= 2.
__device__ __forceinline__ uint64_t sp_perm(uint64_t j, uint64_t d, uint64_t key) {
  const int bits = 64 - __builtin_clzll(d - 1);  // d - 1 >= 1
  const int h = (bits + 1) >> 1;
  const uint64_t mask = (1ull << h) - 1ull;
  uint64_t x = j;
  do {
    uint64_t l = x >> h, r = x & mask;
#pragma unroll
    for (int round = 0; round < 4; ++round) {
      const uint64_t f = sp_mix64(r ^ key ^ ((uint64_t)round << 56)) & mask;
      const uint64_t t = l ^ f;
      l = r;
      r = t;
    }
    x = (l << h) | r;
  } while (x >= d);  // the walk stays inside x's cycle, which contains the start value < d
  return x;
}

__global__ __launch_bounds__(HC_BLOCK) void sp_fill_map(int32_t *__restrict__ loc, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (i < n) loc[i] = SP_UNSEEN;
}

__global__ __launch_bounds__(HC_BLOCK) void sp_init(const int64_t *__restrict__ seeds, int64_t n_seed,
                                                     int64_t num_nodes, int32_t *__restrict__ loc,
                                                     int64_t *__restrict__ sub_to_full, int64_t *__restrict__ ptr,
                                                     int64_t *__restrict__ counts, SpState *__restrict__ st,
                                                     uint64_t rng_seed, const uint64_t *__restrict__ rng_seed_at) {
  const int64_t i = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (i == 0) {
    st->lo = 0;
    st->hi = n_seed;
    st->edges = 0;
    st->key = rng_seed_at ? *rng_seed_at : rng_seed;
    ptr[0] = 0;
    counts[0] = n_seed;
  }
  if (i >= n_seed) return;
  const int64_t s = seeds[i];
  sub_to_full[i] = s;
  if (s >= 0 && s < num_nodes) loc[s] = (int32_t)i;
}

// Sums of a hop's tiles.  `before` (nullable: few tiles) holds the exclusive scan and, behind the last tile, the
// total.
struct SpTiles {
  int32_t *sum;
  int32_t *before;
};

// Sum of the first n tiles, by a whole wave; every lane ends with it.
__device__ __forceinline__ int32_t sp_before(const SpTiles &t, int64_t n, int lane) {
  if (t.before != nullptr) return t.before[n];
  int32_t v = 0;
  for (int64_t i = lane; i < n; i += HC_WAVE) v += t.sum[i];
#pragma unroll
  for (int d = HC_WAVE / 2; d > 0; d >>= 1) v += __shfl_xor(v, d, HC_WAVE);
  return v;
}

__device__ __forceinline__ int64_t sp_tiles_of(int64_t n) { return (n + SP_TILE - 1) / SP_TILE; }

// Exclusive sum over the block's threads (every thread calls it once per launch); *total: the block's.
__device__ __forceinline__ int32_t sp_block_exclusive(int32_t v, int32_t *s_wave, int32_t *total) {
  const int lane = hc_lane(), wave = (int)(threadIdx.x >> 6);
  int32_t x = v;
#pragma unroll
  for (int d = 1; d < HC_WAVE; d <<= 1) {
    const int32_t y = __shfl_up(x, d, HC_WAVE);
    if (lane >= d) x += y;
  }
  if (lane == HC_WAVE - 1) s_wave[wave] = x;
  __syncthreads();
  int32_t base = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < SP_BLOCK / HC_WAVE; ++w) {
    const int32_t t = s_wave[w];
    if (w < wave) base += t;
    sum += t;
  }
  *total = sum;
  return base + x - v;
}

// One block: before[0 .. n] of a hop's row tiles (edges: false) or edge tiles.
__global__ __launch_bounds__(SP_BLOCK) void sp_tile_scan(SpTiles rows, SpTiles edges, const SpState *__restrict__ st,
                                                          int of_edges) {
  __shared__ int32_t s_wave[SP_BLOCK / HC_WAVE];
  const int64_t n_rows = sp_tiles_of(st->hi - st->lo);
  const int64_t n = of_edges ? sp_tiles_of(sp_before(rows, n_rows, hc_lane())) : n_rows;
  const SpTiles t = of_edges ? edges : rows;
  int32_t carry = 0;
  for (int64_t base = 0; base < n; base += SP_BLOCK) {
    const int64_t i = base + threadIdx.x;
    const int32_t v = i < n ? t.sum[i] : 0;
    int32_t total;
    const int32_t x = sp_block_exclusive(v, s_wave, &total);
    if (i < n) t.before[i] = carry + x;
    carry += total;
    __syncthreads();
  }
  if (threadIdx.x == 0) t.before[n] = carry;
}

__global__ __launch_bounds__(SP_BLOCK) void sp_count(const int64_t *__restrict__ indptr,
                                                      const int64_t *__restrict__ sub_to_full,
                                                      const SpState *__restrict__ st, int64_t fanout,
                                                      int64_t num_nodes, int hop, int32_t *__restrict__ loc,
                                                      int32_t *__restrict__ incl, SpTiles rows) {
  __shared__ int32_t s_wave[SP_BLOCK / HC_WAVE];
  const int64_t lo = st->lo, n = st->hi - lo;
  const int64_t i0 = (int64_t)blockIdx.x * SP_TILE + (int64_t)threadIdx.x * SP_ITEMS;
  if ((int64_t)blockIdx.x * SP_TILE >= n) return;
  int64_t full[SP_ITEMS];
  int32_t c[SP_ITEMS];
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) full[k] = i0 + k < n ? sub_to_full[lo + i0 + k] : -1;
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) {
    c[k] = 0;
    if (full[k] >= 0 && full[k] < num_nodes) {
      const int64_t d = indptr[full[k] + 1] - indptr[full[k]];
      c[k] = (int32_t)(d < fanout ? (d < 0 ? 0 : d) : fanout);
      if (hop > 0) loc[full[k]] = (int32_t)(lo + i0 + k);
    }
  }
#pragma unroll
  for (int k = 1; k < SP_ITEMS; ++k) c[k] += c[k - 1];
  int32_t total;
  const int32_t before = sp_block_exclusive(c[SP_ITEMS - 1], s_wave, &total);
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k)
    if (i0 + k < n) incl[i0 + k] = before + c[k];
  if (threadIdx.x == 0) rows.sum[blockIdx.x] = total;
}

__global__ __launch_bounds__(HC_BLOCK) void sp_pick(const int64_t *__restrict__ indptr,
                                                     const int64_t *__restrict__ indices,
                                                     const int64_t *__restrict__ sub_to_full,
                                                     const SpState *__restrict__ st, int64_t fanout,
                                                     int64_t num_nodes, int hop,
                                                     const int32_t *__restrict__ incl, SpTiles rows,
                                                     int32_t *__restrict__ loc, int64_t *__restrict__ ptr,
                                                     int64_t *__restrict__ idx) {
  const int group = sp_group(fanout), side = HC_WAVE / group;             // `side` rows per wave
  const int lane = hc_lane(), in_wave = lane / group, sub = lane - in_wave * group;
  const int64_t lo = st->lo, n = st->hi - lo;
  static_assert(HC_BLOCK <= SP_TILE, "a block's rows lie in two tiles at most");
  const int64_t first_row = (int64_t)blockIdx.x * HC_WAVES_PER_BLOCK * side;
  if (first_row >= n) return;
  const int64_t tile = first_row / SP_TILE;
  int32_t tile_begin = sp_before(rows, tile, lane);
  const int64_t i = first_row + hc_wave_in_block() * side + in_wave;
  if (i >= n || in_wave >= side) return;
  if (i / SP_TILE != tile) tile_begin += rows.sum[tile];
  const int64_t u = lo + i;
  const int32_t in_tile = i % SP_TILE > 0 ? incl[i - 1] : 0;
  const int64_t begin = (int64_t)tile_begin + in_tile;     // slot of the row's first pick inside this hop
  const int32_t c = incl[i] - in_tile;
  const int64_t base = st->edges;
  if (sub == 0) ptr[u + 1] = base + begin + c;
  if (c == 0) return;
  const int64_t full = sub_to_full[u];
  const int64_t first = indptr[full];
  const uint64_t d = (uint64_t)(indptr[full + 1] - first);
  const uint64_t key = sp_mix64(sp_mix64(st->key + (uint64_t)hop) ^ (uint64_t)full);
  for (int64_t j = sub; j < c; j += group) {
    const uint64_t pos = d > (uint64_t)fanout ? sp_perm((uint64_t)j, d, key) : (uint64_t)j;
    const int64_t v = indices[first + (int64_t)pos];
    idx[base + begin + j] = v;
    if (v >= 0 && v < num_nodes) atomicMin(loc + v, SP_PROV + (int32_t)(begin + j));
  }
}

// The owners among a hop's edge slots: bit p % 64 of bits[p / 64], and word_before[p / 64], the owners in front of
// those 64 slots inside their tile.
struct SpOwners {
  unsigned long long *bits;
  int32_t *word_before;
  SpTiles tiles;
};

__global__ __launch_bounds__(SP_BLOCK) void sp_flag(const int64_t *__restrict__ idx, const int32_t *__restrict__ loc,
                                                     const SpState *__restrict__ st, SpTiles rows, int64_t num_nodes,
                                                     SpOwners own) {
  __shared__ int32_t s_wave[SP_BLOCK / HC_WAVE];
  const int lane = hc_lane(), wave = (int)(threadIdx.x >> 6);
  const int64_t hop_edges = sp_before(rows, sp_tiles_of(st->hi - st->lo), lane);
  const int64_t tile0 = (int64_t)blockIdx.x * SP_TILE;
  if (tile0 >= hop_edges) return;
  const int64_t base = st->edges;
  const int64_t w0 = tile0 + (int64_t)wave * SP_ITEMS * HC_WAVE;       // the wave's SP_ITEMS words
  int64_t v[SP_ITEMS];
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) {
    const int64_t p = w0 + k * HC_WAVE + lane;
    v[k] = p < hop_edges ? idx[base + p] : -1;
  }
  unsigned long long b[SP_ITEMS];
  int32_t mine = 0;
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) {
    const int64_t p = w0 + k * HC_WAVE + lane;
    b[k] = __ballot(v[k] >= 0 && v[k] < num_nodes && loc[v[k]] == SP_PROV + (int32_t)p);
    mine += (int32_t)__popcll(b[k]);
  }
  if (lane == 0) s_wave[wave] = mine;
  __syncthreads();
  int32_t before = 0, total = 0;
#pragma unroll
  for (int w = 0; w < SP_BLOCK / HC_WAVE; ++w) {
    const int32_t t = s_wave[w];
    if (w < wave) before += t;
    total += t;
  }
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < SP_ITEMS; ++k) {
      own.bits[w0 / HC_WAVE + k] = b[k];
      own.word_before[w0 / HC_WAVE + k] = before;
      before += (int32_t)__popcll(b[k]);
    }
  }
  if (threadIdx.x == 0) own.tiles.sum[blockIdx.x] = total;
}

__global__ __launch_bounds__(SP_BLOCK) void sp_relabel(int64_t *__restrict__ idx, const int32_t *__restrict__ loc,
                                                        const SpState *__restrict__ st, SpState *__restrict__ next,
                                                        SpTiles rows, int64_t num_nodes, SpOwners own,
                                                        int64_t *__restrict__ sub_to_full,
                                                        int64_t *__restrict__ counts, int hop, int num_hops) {
  __shared__ int32_t s_tile[SP_DIRECT_TILES + 1];
  __shared__ int32_t s_wave[SP_BLOCK / HC_WAVE];
  const int lane = hc_lane();
  const int64_t hop_edges = sp_before(rows, sp_tiles_of(st->hi - st->lo), lane);
  const int64_t tile0 = (int64_t)blockIdx.x * SP_TILE;
  if (tile0 >= hop_edges && blockIdx.x > 0) return;
  const int64_t n_tiles = sp_tiles_of(hop_edges);
  const int32_t *tile_before = own.tiles.before;
  if (tile_before == nullptr) {                            // every block scans the tiles' sums: at most 4096 of them
    const int per = (int)((n_tiles + SP_BLOCK - 1) / SP_BLOCK), t0 = (int)threadIdx.x * per;
    int32_t sum = 0, total;
    for (int t = t0; t < t0 + per && t < n_tiles; ++t) sum += own.tiles.sum[t];
    int32_t run = sp_block_exclusive(sum, s_wave, &total);
    for (int t = t0; t < t0 + per && t < n_tiles; ++t) {
      s_tile[t] = run;
      run += own.tiles.sum[t];
    }
    if (threadIdx.x == 0) s_tile[SP_DIRECT_TILES] = total;
    __syncthreads();
    tile_before = s_tile;
  }
  const int64_t hi = st->hi, base = st->edges;
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // the next hop's state (this hop's is read by the other threads and stays as it is)
    const int64_t fresh = own.tiles.before != nullptr ? tile_before[n_tiles] : s_tile[SP_DIRECT_TILES];
    next->lo = hi;
    next->hi = hi + fresh;
    next->edges = base + hop_edges;
    next->key = st->key;
    counts[hop + 1] = hi + fresh;
    counts[num_hops + 1 + hop] = base + hop_edges;
  }
  int64_t v[SP_ITEMS];
  int32_t t[SP_ITEMS];
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) {
    const int64_t p = tile0 + k * SP_BLOCK + threadIdx.x;
    v[k] = p < hop_edges ? idx[base + p] : -1;
  }
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) t[k] = v[k] >= 0 && v[k] < num_nodes ? loc[v[k]] : -1;
#pragma unroll
  for (int k = 0; k < SP_ITEMS; ++k) {
    const int64_t p = tile0 + k * SP_BLOCK + threadIdx.x;
    if (p >= hop_edges) continue;
    int64_t id = t[k];                            // -1: not a node of the graph
    if (t[k] >= SP_PROV) {
      const int32_t q = t[k] - SP_PROV;           // the owning edge slot of this hop
      const unsigned long long below = own.bits[q / HC_WAVE] & ((1ull << (q % HC_WAVE)) - 1ull);
      id = hi + tile_before[q / SP_TILE] + own.word_before[q / HC_WAVE] + (int32_t)__popcll(below);
      if (q == (int32_t)p) sub_to_full[id] = v[k];
    }
    idx[base + p] = id;
  }
}

__global__ __launch_bounds__(HC_BLOCK) void sp_reset(const int64_t *__restrict__ sub_to_full,
                                                      const SpState *__restrict__ st, int64_t num_nodes,
                                                      int32_t *__restrict__ loc, int64_t node_cap) {
  const int64_t i = (int64_t)blockIdx.x * HC_BLOCK + threadIdx.x;
  if (i >= node_cap || i >= st->hi) return;
  const int64_t v = sub_to_full[i];
  if (v >= 0 && v < num_nodes) loc[v] = SP_UNSEEN;
}

struct SpCaps {
  int64_t rows[HC_SAMPLE_MAX_HOPS];   // frontier bound per hop
  int64_t edges[HC_SAMPLE_MAX_HOPS];  // edge bound per hop
  int64_t max_rows, max_edges, total_rows, total_edges, total_nodes;
  bool ok;
};

SpCaps sp_caps(int64_t n_seed, const int64_t *fanout, int num_hops, int64_t num_nodes) {
  SpCaps c{};
  c.ok = num_hops >= 1 && num_hops <= HC_SAMPLE_MAX_HOPS && n_seed >= 0 && fanout != nullptr;
  if (!c.ok) return c;
  int64_t rows = n_seed;
  c.total_nodes = n_seed;
  for (int k = 0; k < num_hops; ++k) {
    if (fanout[k] < 1 || fanout[k] > (1 << 20)) {
      c.ok = false;
      return c;
    }
    c.rows[k] = rows;
    c.edges[k] = rows * fanout[k];
    if (c.edges[k] >= (int64_t)SP_PROV - 1) {
      c.ok = false;
      return c;
    }
    c.total_rows += rows;
    c.total_edges += c.edges[k];
    if (rows > c.max_rows) c.max_rows = rows;
    if (c.edges[k] > c.max_edges) c.max_edges = c.edges[k];
    // new nodes of a hop: at most its edges, and at most the graph
    rows = c.edges[k];
    if (num_nodes > 0 && rows > num_nodes) rows = num_nodes;
    c.total_nodes += rows;
  }
  if (num_nodes > 0 && c.total_nodes > num_nodes) c.total_nodes = num_nodes > n_seed ? num_nodes : n_seed;
  if (c.total_nodes >= (int64_t)SP_PROV) c.ok = false;
  return c;
}

struct SpLayout {
  size_t state, incl, row_sum, row_before, bits, word_before, edge_sum, edge_before, total;
};

inline int64_t sp_tiles(int64_t n) { return (n + SP_TILE - 1) / SP_TILE; }

SpLayout sp_layout(const SpCaps &c) {
  SpLayout l{};
  size_t off = 0;
  const auto take = [&off](size_t bytes) {
    const size_t here = off;
    off += hc_align_up(bytes, 256);
    return here;
  };
  l.state = take(sizeof(SpState) * (HC_SAMPLE_MAX_HOPS + 1));      // one state per hop and the final one
  l.incl = take((size_t)(c.max_rows + 1) * 4);
  l.row_sum = take((size_t)(sp_tiles(c.max_rows) + 1) * 4);
  l.row_before = take((size_t)(sp_tiles(c.max_rows) + 1) * 4);
  l.bits = take((size_t)sp_tiles(c.max_edges) * (SP_TILE / HC_WAVE) * 8);
  l.word_before = take((size_t)sp_tiles(c.max_edges) * (SP_TILE / HC_WAVE) * 4);
  l.edge_sum = take((size_t)(sp_tiles(c.max_edges) + 1) * 4);
  l.edge_before = take((size_t)(sp_tiles(c.max_edges) + 1) * 4);
  l.total = off;
  return l;
}

inline unsigned sp_blocks(int64_t n) { return (unsigned)((n + HC_BLOCK - 1) / HC_BLOCK); }

}  // namespace

extern "C" int hc_sample_capacity(int64_t n_seed, const int64_t *fanout, int num_hops, int64_t num_nodes,
                                  int64_t *max_rows, int64_t *max_edges, int64_t *max_nodes) {
  const SpCaps c = sp_caps(n_seed, fanout, num_hops, num_nodes);
  if (!c.ok) return HC_EINVAL;
  if (max_rows) *max_rows = c.total_rows;
  if (max_edges) *max_edges = c.total_edges;
  if (max_nodes) *max_nodes = c.total_nodes;
  return HC_OK;
}

extern "C" size_t hc_sample_workspace_bytes(int64_t n_seed, const int64_t *fanout, int num_hops,
                                            int64_t num_nodes) {
  const SpCaps c = sp_caps(n_seed, fanout, num_hops, num_nodes);
  if (!c.ok) return 0;
  return sp_layout(c).total;
}

extern "C" int hc_sample_map_init(int32_t *node_map, int64_t num_nodes, void *stream) {
  HC_REQUIRE(num_nodes >= 0);
  if (num_nodes == 0) return HC_OK;
  HC_REQUIRE(node_map != nullptr);
  if (!hc_grid_ok(sp_blocks(num_nodes))) return HC_EUNSUPPORTED;
  sp_fill_map<<<dim3(sp_blocks(num_nodes)), dim3(HC_BLOCK), 0, static_cast<hipStream_t>(stream)>>>(node_map,
                                                                                                  num_nodes);
  return hc_launch_status();
}

namespace {

int sample_layers_impl(const int64_t *indptr, const int64_t *indices, int64_t num_nodes, const int64_t *seeds,
                       int64_t n_seed, const int64_t *fanout, int num_hops, uint64_t rng_seed,
                       const uint64_t *rng_seed_at, int32_t *node_map, int64_t *ptr, int64_t *idx,
                       int64_t *sub_to_full, int64_t *counts, void *workspace, size_t workspace_bytes,
                       void *stream) {
  HC_REQUIRE(num_nodes > 0 && n_seed > 0);
  HC_REQUIRE(indptr && indices && seeds && node_map && ptr && idx && sub_to_full && counts);
  const SpCaps c = sp_caps(n_seed, fanout, num_hops, num_nodes);
  if (!c.ok) return HC_EUNSUPPORTED;
  const SpLayout l = sp_layout(c);
  if (!workspace || workspace_bytes < l.total) return HC_EWORKSPACE;
  if (!hc_grid_ok(sp_blocks(c.max_edges)) || !hc_grid_ok(sp_blocks(c.max_rows * SP_GROUP)) ||
      !hc_grid_ok(sp_blocks(c.total_nodes)))
    return HC_EUNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char *w = static_cast<char *>(workspace);
  SpState *states = reinterpret_cast<SpState *>(w + l.state);
  int32_t *incl = reinterpret_cast<int32_t *>(w + l.incl);
  const dim3 bl(HC_BLOCK), tl(SP_BLOCK);

  sp_init<<<dim3(sp_blocks(n_seed)), bl, 0, s>>>(seeds, n_seed, num_nodes, node_map, sub_to_full, ptr, counts, states,
                                                 rng_seed, rng_seed_at);
  for (int k = 0; k < num_hops; ++k) {
    const int64_t cap = c.rows[k], ecap = c.edges[k];
    const int64_t row_tiles = sp_tiles(cap), edge_tiles = sp_tiles(ecap);
    const SpState *st = states + k;
    SpTiles rows{reinterpret_cast<int32_t *>(w + l.row_sum), reinterpret_cast<int32_t *>(w + l.row_before)};
    SpOwners own{reinterpret_cast<unsigned long long *>(w + l.bits), reinterpret_cast<int32_t *>(w + l.word_before),
                 {reinterpret_cast<int32_t *>(w + l.edge_sum), reinterpret_cast<int32_t *>(w + l.edge_before)}};
    if (row_tiles <= SP_DIRECT_TILES) rows.before = nullptr;
    if (edge_tiles <= SP_DIRECT_TILES) own.tiles.before = nullptr;
    sp_count<<<dim3((unsigned)row_tiles), tl, 0, s>>>(indptr, sub_to_full, st, fanout[k], num_nodes, k, node_map, incl,
                                                      rows);
    if (rows.before != nullptr) sp_tile_scan<<<dim3(1), tl, 0, s>>>(rows, own.tiles, st, 0);
    const int64_t pick_rows = (int64_t)HC_WAVES_PER_BLOCK * (HC_WAVE / sp_group(fanout[k]));
    sp_pick<<<dim3((unsigned)((cap + pick_rows - 1) / pick_rows)), bl, 0, s>>>(indptr, indices, sub_to_full, st, fanout[k], num_nodes,
                                                          k, incl, rows, node_map, ptr, idx);
    sp_flag<<<dim3((unsigned)edge_tiles), tl, 0, s>>>(idx, node_map, st, rows, num_nodes, own);
    if (own.tiles.before != nullptr) sp_tile_scan<<<dim3(1), tl, 0, s>>>(rows, own.tiles, st, 1);
    sp_relabel<<<dim3((unsigned)edge_tiles), tl, 0, s>>>(idx, node_map, st, states + k + 1, rows, num_nodes, own,
                                                        sub_to_full, counts, k, num_hops);
    if (hc_launch_status() != HC_OK) return HC_ELAUNCH;
  }
  const SpState *st = states + num_hops;
  sp_reset<<<dim3(sp_blocks(c.total_nodes)), bl, 0, s>>>(sub_to_full, st, num_nodes, node_map, c.total_nodes);
  return hc_launch_status();
}

}  // namespace

extern "C" int hc_sample_layers(const int64_t *indptr, const int64_t *indices, int64_t num_nodes,
                                const int64_t *seeds, int64_t n_seed, const int64_t *fanout, int num_hops,
                                uint64_t rng_seed, int32_t *node_map, int64_t *ptr, int64_t *idx,
                                int64_t *sub_to_full, int64_t *counts, void *workspace, size_t workspace_bytes,
                                void *stream) {
  return sample_layers_impl(indptr, indices, num_nodes, seeds, n_seed, fanout, num_hops, rng_seed, nullptr, node_map,
                            ptr, idx, sub_to_full, counts, workspace, workspace_bytes, stream);
}

extern "C" int hc_sample_layers_seed_at(const int64_t *indptr, const int64_t *indices, int64_t num_nodes,
                                        const int64_t *seeds, int64_t n_seed, const int64_t *fanout, int num_hops,
                                        const uint64_t *rng_seed_at, int32_t *node_map, int64_t *ptr,
                                        int64_t *idx, int64_t *sub_to_full, int64_t *counts, void *workspace,
                                        size_t workspace_bytes, void *stream) {
  HC_REQUIRE(rng_seed_at != nullptr);
  return sample_layers_impl(indptr, indices, num_nodes, seeds, n_seed, fanout, num_hops, 0, rng_seed_at, node_map,
                            ptr, idx, sub_to_full, counts, workspace, workspace_bytes, stream);
}
