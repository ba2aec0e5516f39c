// Shared device/host helpers for the gfx950 kernels (wave64 only).
#pragma once

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "hiscache_hip.h"

#define HC_WAVE 64
#define HC_BLOCK 256
#define HC_WAVES_PER_BLOCK (HC_BLOCK / HC_WAVE)

#define HC_REQUIRE(cond) \
  do {                   \
    if (!(cond)) return HC_EINVAL; \
  } while (0)

static inline int hc_launch_status() {
  return hipGetLastError() == hipSuccess ? HC_OK : HC_ELAUNCH;
}

static inline size_t hc_align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

// Grid limit for a 1-D launch: gridDim.x * blockDim.x must stay below 2^32 (blocks of up to
// 1024 threads are used by the scan kernel, so the bound is taken for those).
static inline bool hc_grid_ok(int64_t blocks) { return blocks > 0 && blocks <= 0xffffffffLL / HC_BLOCK; }

// feature_tiers.hip: the plain row gather of a matrix in device memory, several rows per wave
// (hc_gather_rows hands such calls over; arguments are checked there).
__attribute__((visibility("hidden"))) int hc_gather_rows_device(const void *src, int src_dtype, int64_t n_rows, const int64_t *ids, const uint8_t *mask,
                          void *dst, int dst_dtype, int64_t n, int64_t F, hipStream_t st);

// feature_tiers.hip: hc_fixup_rows' launch (64 rows examined per wave, the few that differ read or cleared).
__attribute__((visibility("hidden"))) int hc_fixup_rows_chunked(const void *src, int src_dtype, int64_t n_rows,
                                                                const int64_t *ids, const uint8_t *need,
                                                                const uint8_t *have, void *dst, int dst_dtype,
                                                                int64_t n, int64_t F, hipStream_t st);

// edge_grad.hip: the gradient of the edge weights (hc_aggr_bwd hands over; arguments are checked there).
__attribute__((visibility("hidden"))) int hc_edge_grad(const int64_t *ptr, const int64_t *idx, const float *g,
                                                       const int64_t *hmap, const void *vin, int in_dtype,
                                                       float *edge_grad, int64_t E, int64_t R, int64_t F,
                                                       int64_t n_head, hipStream_t st);

#ifdef __HIPCC__

__device__ __forceinline__ int hc_lane() { return (int)(threadIdx.x & (HC_WAVE - 1)); }

// Index of this wave inside its block, forced into a scalar register so that
// everything derived from it (row id, row bounds) is wave-uniform.
__device__ __forceinline__ int hc_wave_in_block() {
  return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

__device__ __forceinline__ int64_t hc_readlane64(int64_t v, int lane) {
  int lo = __builtin_amdgcn_readlane((int)(uint32_t)(uint64_t)v, lane);
  int hi = __builtin_amdgcn_readlane((int)(uint32_t)((uint64_t)v >> 32), lane);
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint64_t)(uint32_t)lo);
}

__device__ __forceinline__ int64_t hc_uniform64(int64_t v) {
  int lo = __builtin_amdgcn_readfirstlane((int)(uint32_t)(uint64_t)v);
  int hi = __builtin_amdgcn_readfirstlane((int)(uint32_t)((uint64_t)v >> 32));
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | (uint64_t)(uint32_t)lo);
}

__device__ __forceinline__ float hc_readlane_f(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Workgroups are handed to the 8 XCDs round-robin (workgroup i runs on XCD i % 8) and every XCD
// has its own L2.  This maps the hardware block index to a logical one so that an XCD works on
// runs of CHUNK consecutive logical blocks: neighbouring rows or sources, which tend to touch the
// same index lines and the same data, then share an L2.  The runs of the 8 XCDs are interleaved
// (XCD x takes run x of every group of 8 runs), so that work whose cost drifts along the block
// range -- rows sorted by degree, layers with different fan-outs -- stays balanced over the XCDs.
// A bijection of [0, n); blocks behind the last full group keep their index.
#define HC_NUM_XCD 8
template <int CHUNK>
__device__ __forceinline__ int64_t hc_xcd_block(int64_t bid, int64_t n) {
  constexpr uint32_t GROUP = (uint32_t)HC_NUM_XCD * CHUNK;       // a power of two; a grid has less than 2^24 blocks
  const uint32_t b = (uint32_t)bid, in = b % GROUP, first = b - in;
  if (first + GROUP > (uint32_t)n) return bid;
  return first + (in % HC_NUM_XCD) * CHUNK + in / HC_NUM_XCD;
}

// Butterfly sum over the 64 lanes, partner distance 32,16,8,4,2,1.  Every lane
// ends with the same bits (fp add is commutative), and the order is the one
// the oracle reproduces.
__device__ __forceinline__ float hc_wave_sum_butterfly(float v) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) v = v + __shfl_xor(v, d, HC_WAVE);
  return v;
}

// The calling block arrives at a counter that `of` blocks take (every thread of them calls this).  True in every
// thread of the block that arrives last, which then sees what all of them had stored; the counter is zero again.
// Every wave waits for its own stores in front of the barrier: a release of workgroup scope waits for the LDS alone,
// and the device-scope release that thread 0 makes behind the barrier waits for its own wave's stores only, before
// it writes the die's L2 back.  (One release of device scope per wave would do as well, at one write-back each.)
__device__ __forceinline__ bool hc_arrives_last(unsigned *ticket, unsigned of, int *s_flag) {
  constexpr int VMCNT_0 = 0x0f70;      // s_waitcnt: vmcnt 0, the other counters at their largest
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(VMCNT_0);
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    const unsigned t = atomicAdd(ticket, 1u);
    *s_flag = t == of - 1u ? 1 : 0;
    if (t == of - 1u) atomicExch(ticket, 0u);
  }
  __syncthreads();
  if (*s_flag == 0) return false;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  return true;
}

// ---- element conversion ----------------------------------------------------
template <typename T>
__device__ __forceinline__ float hc_to_f32(T v);
template <>
__device__ __forceinline__ float hc_to_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ float hc_to_f32<__half>(__half v) { return __half2float(v); }
template <>
__device__ __forceinline__ float hc_to_f32<__hip_bfloat16>(__hip_bfloat16 v) {
  return __bfloat162float(v);
}

template <typename T>
__device__ __forceinline__ T hc_from_f32(float v);
template <>
__device__ __forceinline__ float hc_from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ __half hc_from_f32<__half>(float v) { return __float2half_rn(v); }
template <>
__device__ __forceinline__ __hip_bfloat16 hc_from_f32<__hip_bfloat16>(float v) {
  return __float2bfloat16(v);
}

// ---- vector load of VEC consecutive elements, widened to fp32 ---------------
template <int BYTES>
struct hc_raw;
template <>
struct hc_raw<2> { typedef uint16_t type; };
template <>
struct hc_raw<4> { typedef uint32_t type; };
template <>
struct hc_raw<8> { typedef uint2 type; };
template <>
struct hc_raw<16> { typedef uint4 type; };

template <typename T, int VEC>
struct hc_vec {
  typedef typename hc_raw<sizeof(T) * VEC>::type raw_t;
  union U {
    raw_t raw;
    T e[VEC];
    __device__ U() {}
  };
  // p must be aligned to sizeof(T) * VEC
  __device__ __forceinline__ static void load(const T *p, float (&out)[VEC]) {
    U u;
    u.raw = *reinterpret_cast<const raw_t *>(p);
#pragma unroll
    for (int i = 0; i < VEC; ++i) out[i] = hc_to_f32<T>(u.e[i]);
  }
  __device__ __forceinline__ static void store(T *p, const float (&in)[VEC]) {
    U u;
#pragma unroll
    for (int i = 0; i < VEC; ++i) u.e[i] = hc_from_f32<T>(in[i]);
    *reinterpret_cast<raw_t *>(p) = u.raw;
  }
  // Same load / store with the non-temporal hint: rows that are read or written once should not
  // displace the index and map lines that are reused.
  typedef uint32_t nt_t __attribute__((ext_vector_type(sizeof(T) * VEC >= 4 ? sizeof(T) * VEC / 4 : 1)));
  __device__ __forceinline__ static void load_nt(const T *p, float (&out)[VEC]) {
    if constexpr (sizeof(T) * VEC >= 4) {
      union N {
        nt_t raw;
        T e[VEC];
        __device__ N() {}
      } u;
      u.raw = __builtin_nontemporal_load(reinterpret_cast<const nt_t *>(p));
#pragma unroll
      for (int i = 0; i < VEC; ++i) out[i] = hc_to_f32<T>(u.e[i]);
    } else {
      load(p, out);
    }
  }
  __device__ __forceinline__ static void store_nt(T *p, const float (&in)[VEC]) {
    if constexpr (sizeof(T) * VEC >= 4) {
      union N {
        nt_t raw;
        T e[VEC];
        __device__ N() {}
      } u;
#pragma unroll
      for (int i = 0; i < VEC; ++i) u.e[i] = hc_from_f32<T>(in[i]);
      __builtin_nontemporal_store(u.raw, reinterpret_cast<nt_t *>(p));
    } else {
      store(p, in);
    }
  }
};

// ---- pieces of a row whose base address is a wave-uniform integer ------------
// Loads through an explicit global pointer (base in scalar registers, 32-bit byte offset per lane).  A pointer
// made from an integer is otherwise taken as generic: flat loads, which also occupy the LDS counter, so that a
// wave can only wait for all of them at once.  `raw_t` keeps the element type until the value is used.
#define HC_GLOBAL __attribute__((address_space(1)))
template <int BYTES>
struct hc_piece_raw;
template <>
struct hc_piece_raw<2> { typedef uint16_t type; };
template <>
struct hc_piece_raw<4> { typedef uint32_t type; };
template <>
struct hc_piece_raw<8> { typedef uint32_t type __attribute__((ext_vector_type(2))); };
template <>
struct hc_piece_raw<16> { typedef uint32_t type __attribute__((ext_vector_type(4))); };

template <typename T, int VEC>
struct hc_piece {
  typedef typename hc_piece_raw<sizeof(T) * VEC>::type raw_t;
  // base + byte must be aligned to sizeof(T) * VEC
  template <bool NT>
  __device__ __forceinline__ static raw_t load(int64_t base, uint32_t byte) {
    const HC_GLOBAL char *p = (const HC_GLOBAL char *)base + byte;
    if constexpr (NT) return __builtin_nontemporal_load((const HC_GLOBAL raw_t *)p);
    else return *(const HC_GLOBAL raw_t *)p;
  }
  __device__ __forceinline__ static float widen(const raw_t &r, int i) {
    if constexpr (std::is_same<T, float>::value) {
      if constexpr (VEC == 1) return __uint_as_float(r);
      else return __uint_as_float(r[i]);
    } else {
      uint32_t w;
      if constexpr (VEC <= 2) w = r;
      else w = r[i >> 1];
      if constexpr (std::is_same<T, __hip_bfloat16>::value) {
        return __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
      } else {
        const uint16_t h = (uint16_t)((i & 1) ? (w >> 16) : w);
        return __half2float(__builtin_bit_cast(__half, h));
      }
    }
  }
};

// One word (or half word) of a row at a wave-uniform 32-bit offset from a matrix of less than 4 GiB: a buffer
// load takes the row's offset from a scalar register and the lane's from a vector register, which leaves one
// v_readlane per row as address arithmetic.
typedef __amdgpu_buffer_rsrc_t hc_buffer;
__device__ __forceinline__ hc_buffer hc_make_buffer(const void *base, uint32_t bytes = 0xffffffffu) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, bytes, 0x00027000);
}
template <typename RAW>
__device__ __forceinline__ RAW hc_buffer_load(hc_buffer b, uint32_t lane_byte, uint32_t row_byte) {
  if constexpr (sizeof(RAW) == 2) return __builtin_amdgcn_raw_buffer_load_b16(b, lane_byte, row_byte, 0);
  else return __builtin_amdgcn_raw_buffer_load_b32(b, lane_byte, row_byte, 0);
}

// A piece of a row that has a descriptor of its own, with the non-temporal hint; behind its end: zeros.
template <typename RAW>
__device__ __forceinline__ RAW hc_buffer_load_nt(hc_buffer b, uint32_t lane_byte) {
  constexpr int NT = 2;
  if constexpr (sizeof(RAW) == 2) return __builtin_bit_cast(RAW, __builtin_amdgcn_raw_buffer_load_b16(b, lane_byte, 0, NT));
  else if constexpr (sizeof(RAW) == 4) return __builtin_bit_cast(RAW, __builtin_amdgcn_raw_buffer_load_b32(b, lane_byte, 0, NT));
  else if constexpr (sizeof(RAW) == 8) return __builtin_bit_cast(RAW, __builtin_amdgcn_raw_buffer_load_b64(b, lane_byte, 0, NT));
  else return __builtin_bit_cast(RAW, __builtin_amdgcn_raw_buffer_load_b128(b, lane_byte, 0, NT));
}

// Store VEC consecutive fp32 values (VEC may exceed one 16-byte store).
template <int VEC>
__device__ __forceinline__ void hc_store_f32(float *p, const float (&in)[VEC]) {
  if constexpr (VEC <= 4) {
    hc_vec<float, VEC>::store(p, in);
  } else {
#pragma unroll
    for (int q = 0; q < VEC / 4; ++q) {
      const float t[4] = {in[4 * q], in[4 * q + 1], in[4 * q + 2], in[4 * q + 3]};
      hc_vec<float, 4>::store(p + 4 * q, t);
    }
  }
}

// Same with the non-temporal hint (output rows that this launch does not read again).
template <int VEC>
__device__ __forceinline__ void hc_store_f32_nt(float *p, const float (&in)[VEC]) {
  if constexpr (VEC <= 4) {
    hc_vec<float, VEC>::store_nt(p, in);
  } else {
#pragma unroll
    for (int q = 0; q < VEC / 4; ++q) {
      const float t[4] = {in[4 * q], in[4 * q + 1], in[4 * q + 2], in[4 * q + 3]};
      hc_vec<float, 4>::store_nt(p + 4 * q, t);
    }
  }
}

#endif  // __HIPCC__
