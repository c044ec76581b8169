// Device-side helpers shared by the gfx950 quantized-matmul kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include "../../include/qmm_hip.h"

namespace qmm {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(8))) int i32x8;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;

constexpr int kWave = 64;

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t b) {
  return __uint_as_float(b << 16);
}

// float32 -> bf16 bits, round to nearest even (v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
  bf16x2 t;
  t[0] = (__bf16)f;
  t[1] = (__bf16)0.0f;
  return __builtin_bit_cast(uint32_t, t) & 0xFFFFu;
}

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2 t;
  t[0] = (__bf16)lo;
  t[1] = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, t);
}

__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
  _Float16 h = (_Float16)f;
  return (uint32_t)__builtin_bit_cast(uint16_t, h);
}

__device__ __forceinline__ float f16_bits_to_f32(uint32_t b) {
  return (float)__builtin_bit_cast(_Float16, (uint16_t)b);
}

// One scale / bias table entry as float32 (exact widening).
template <int TAB>
__device__ __forceinline__ float load_table(const void* p, int64_t i) {
  if constexpr (TAB == QMM_F32) {
    return static_cast<const float*>(p)[i];
  } else if constexpr (TAB == QMM_BF16) {
    return bf16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
  } else {
    return f16_bits_to_f32(static_cast<const uint16_t*>(p)[i]);
  }
}

__device__ __forceinline__ float load_table_rt(const void* p, int64_t i, int tab) {
  if (tab == QMM_F32) return load_table<QMM_F32>(p, i);
  if (tab == QMM_BF16) return load_table<QMM_BF16>(p, i);
  return load_table<QMM_F16>(p, i);
}

// Cache policy of a buffer store that does not stay in the L2 of its XCD (sc1).
constexpr int kWriteThrough = 16;

// Are the float32 sums [R][N] of a split stored sixteen bytes a lane (32-bit offsets)?
__host__ __device__ inline bool wide_sums(int64_t R, int64_t N) { return N % 4 == 0 && R * N < (1 << 29); }

__device__ __forceinline__ void store_out(void* y, int64_t i, float v, int yd) {
  if (yd == QMM_BF16) {
    static_cast<uint16_t*>(y)[i] = (uint16_t)f32_to_bf16_bits(v);
  } else if (yd == QMM_F32) {
    static_cast<float*>(y)[i] = v;
  } else {
    static_cast<uint16_t*>(y)[i] = (uint16_t)f32_to_f16_bits(v);
  }
}

// E8M0 byte -> 2^(e-127) as float32.  Byte 0 is the subnormal 2^-127 and byte
// 255 is NaN, as in the OCP MX specification.
__device__ __forceinline__ float e8m0_to_f32(uint32_t e) {
  uint32_t bits = e << 23;
  if (e == 0u) bits = 0x00400000u;
  if (e == 255u) bits = 0x7FC00000u;
  return __uint_as_float(bits);
}

// E2M1 code (4 bits, bit 3 = sign) -> float32, exact.
__device__ __forceinline__ float e2m1_to_f32(uint32_t c) {
  // magnitudes 0, .5, 1, 1.5, 2, 3, 4, 6 as bf16 high bytes+: build f32 bits
  const uint32_t m = c & 7u;
  // normal (m >= 2): exponent (m>>1) with bias 1, mantissa bit (m&1);
  // m == 1 is the subnormal 0.5; m == 0 is zero.
  uint32_t bits;
  if (m >= 2u) bits = ((126u + (m >> 1)) << 23) | ((m & 1u) << 22);
  else bits = m ? 0x3F000000u : 0u;
  return __uint_as_float(bits | ((c & 8u) << 28));
}

// v_perm_b32: bytes 0-3 of the selector index come from `lo`, 4-7 from `hi`.
__device__ __forceinline__ uint32_t byte_perm(uint32_t hi, uint32_t lo, uint32_t sel) {
  return __builtin_amdgcn_perm(hi, lo, sel);
}

__host__ __device__ constexpr int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// ---- the row tiles of a grouped product --------------------------------------
// Rows [offsets[e], offsets[e+1]) belong to expert e and are cut into tiles of
// `tile_rows` that never straddle two experts.  Which expert and which of its
// tiles is row tile `tile_m` of the whole product?  The wavefront looks at 64
// experts at a time, one a lane (two coalesced loads, a prefix sum over the
// lanes and a ballot), so that the search costs a few memory round trips
// whatever the number of experts -- walked one expert after the other it cost
// one round trip an expert in every workgroup's prologue.  Offsets are forced
// into [0, R] and non-decreasing whatever the array holds.  Every lane of the
// wavefront must be active; the results are the same in all of them.
struct RowTile {
  int e, lo, hi, idx;    // expert, its rows [lo, hi), the tile's number inside the expert
  int m_tiles;           // row tiles of the whole product
  bool found;            // false: tile_m is past the last tile
};

__device__ __forceinline__ RowTile find_row_tile(const int32_t* offsets, int E, int R, int tile_rows, int tile_m) {
  RowTile r{0, 0, 0, 0, 0, false};
  const int lane = (int)(threadIdx.x & 63);
  int base = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int i = e0 + lane;
    int lo = 0, hi = 0;
    if (i < E) {
      lo = offsets[i];
      hi = offsets[i + 1];
      lo = lo < 0 ? 0 : (lo > R ? R : lo);
      hi = hi < lo ? lo : (hi > R ? R : hi);
    }
    const int tiles = (hi - lo + tile_rows - 1) / tile_rows;
    int incl = tiles;                               // tiles of experts e0 .. e0 + lane
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    const int total = __shfl(incl, 63, 64);
    if (!r.found && tile_m >= base && tile_m < base + total) {
      const unsigned long long past = __ballot(base + incl > tile_m);    // lanes at or after the tile's expert
      const int L = __ffsll((long long)past) - 1;
      r.e = e0 + L;
      r.lo = __shfl(lo, L, 64);
      r.hi = __shfl(hi, L, 64);
      r.idx = tile_m - base - __shfl(incl - tiles, L, 64);
      r.found = true;
    }
    base += total;
  }
  r.e = __builtin_amdgcn_readfirstlane(r.e);
  r.lo = __builtin_amdgcn_readfirstlane(r.lo);
  r.hi = __builtin_amdgcn_readfirstlane(r.hi);
  r.idx = __builtin_amdgcn_readfirstlane(r.idx);
  r.m_tiles = __builtin_amdgcn_readfirstlane(base);
  return r;
}

// ---- rows that no expert covers ------------------------------------------------
// A grouped product leaves the rows outside its offsets alone.  For a caller that
// hands over fresh memory they are set to zero here, a wavefront a row, by
// workgroups beside those that re-lay the activations, or by a launch of its own
// where a product has no such launch.  (Every row was zeroed ahead of the product
// before, none of which stayed: a launch of 7.3 us for 1024 x 14336 bf16 results,
// whose product over eight experts takes 172 us with it and 170 without: most of
// the pause comes back as a slower product.)
struct ClearArgs {
  void* y;                      // [R][N], null: nothing is cleared
  const int32_t* row_offsets;   // [E+1]
  int R, E;
  int64_t row_bytes;
};

// Row `row` (the same for the wavefront, every lane active): the offsets are read as find_row_tile reads them.
__device__ __forceinline__ void clear_row_outside(const ClearArgs& c, int row) {
  const int lane = (int)(threadIdx.x & 63);
  for (int e0 = 0; e0 < c.E; e0 += 64) {
    const int i = e0 + lane;
    bool in = false;
    if (i < c.E) {
      int lo = c.row_offsets[i], hi = c.row_offsets[i + 1];
      lo = lo < 0 ? 0 : lo;
      hi = hi < lo ? lo : hi;
      in = row >= lo && row < hi;
    }
    if (__ballot(in)) return;
  }
  char* p = static_cast<char*>(c.y) + (int64_t)row * c.row_bytes;
  if (((reinterpret_cast<uintptr_t>(p) | (uintptr_t)c.row_bytes) & 15u) == 0) {
    for (int64_t i = lane; i < c.row_bytes / 16; i += 64) reinterpret_cast<u32x4*>(p)[i] = u32x4{0u, 0u, 0u, 0u};
  } else {
    for (int64_t i = lane; i < c.row_bytes / 2; i += 64) reinterpret_cast<uint16_t*>(p)[i] = 0;
  }
}

// ---- host-side helpers ------------------------------------------------------

// Experiment switches (kernel overrides used while measuring).  The shipped
// library reads no environment: they exist only in a build with
// -DQMM_EXPERIMENTS.
inline const char* experiment_env(const char* name) {
#ifdef QMM_EXPERIMENTS
  return getenv(name);
#else
  (void)name;
  return nullptr;
#endif
}

// The status of the last failed launch set-up on this thread (hipSuccess when
// none); the C ABI turns it into QMM_ERR_HIP and clears it.
inline hipError_t& setup_error() {
  static thread_local hipError_t e = hipSuccess;
  return e;
}

// Raises kernel KERN's dynamic-LDS limit to MOST, the largest that any launch of it
// asks for.  The HIP call is made once per process (the initialisation of a
// function-local static is thread-safe) and its status is kept: every later call
// reports the same status, so a launch behind a failed set-up is never attempted.
// Returns true when the limit is set.
template <auto KERN, size_t MOST>
inline bool lds_limit() {
  static const hipError_t rc = hipFuncSetAttribute(
      reinterpret_cast<const void*>(KERN), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MOST);
  if (rc != hipSuccess) setup_error() = rc;
  return rc == hipSuccess;
}

// zeroes in the rows that no expert covers, in a launch of its own (qmm_util.hip)
void clear_rows_dispatch(const ClearArgs& c, hipStream_t st);

// y = the splits' float32 sums [splits][R][N], added in order and rounded once (qmm_util.hip)
void split_sum_dispatch(const float* part, void* y, int y_dtype, int64_t R, int64_t N, int splits,
                        const int32_t* row_offsets, int64_t E, const int32_t* out_idx, hipStream_t st);

}  // namespace qmm
