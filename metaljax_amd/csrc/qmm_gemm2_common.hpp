// Pieces shared by the prefill-regime kernels: tile constants, the LDS layout
// of a dequantized weight tile, the kernel arguments and the dequantization of
// one 16-byte piece.
#pragma once

#include "qmm_common.hpp"

namespace qmm {

namespace g2 {

constexpr int BN = 128, BK = 64;
constexpr int kRowBytes = BK * 2;                 // bf16 tile row
constexpr int kStage = BN * kRowBytes;            // 16 KB

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* p, int64_t bytes) {
  const uint32_t n = bytes > 0xFFFFFFFFll ? 0xFFFFFFFFu : (uint32_t)bytes;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, n, 0x00020000);
}

__device__ __forceinline__ void lds_barrier() {   // orders LDS traffic only; global loads stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A bf16 tile row is 128 bytes = half of the 64 banks, so the parity of the
// row picks the half and 16-byte piece p of row r sits at p ^ ((r >> 1) & 7):
// the 16 lanes of one pass of a ds_read_b128 / ds_write_b128 (16 consecutive
// rows of one piece, or 8 rows x 2 halves of 4 pieces) then touch every bank
// once.  (With p ^ (r & 7) rows r and r + 8 shared their banks: every fragment
// read took two passes.)
__device__ __forceinline__ int swz(int row, int piece) {
  return row * kRowBytes + ((piece ^ ((row >> 1) & 7)) << 4);
}

// ---------------------------------------------------------------------------
struct Gemm2Args {
  const void* ax;        // re-laid activations
  const uint32_t* w;     // [E, N, K*bits/32]
  const void* s;         // [E, N, K/gs]
  const void* b;
  void* y;               // [R, N]
  const int32_t* row_offsets;   // [E+1] or null
  const int32_t* out_idx;       // optional row scatter for y
  int R, N, K, E, Rp;
  int gs, tab, y_dtype;
  int m_tiles;
  int tabfast;           // general kernel: float32 tables of groups of 32, fetched as windows
  int tab_ok, tab_odd;   // split-role kernel: tables start on dwords; their rows may start inside one
  int tile_rows;         // split-role kernel: rows a tile may hold (128 or 256)
  int splits;            // split-role kernel, dense (else 1): workgroups that share a tile's K ...
  float* part;           // ... and leave their float32 sums here, [splits][R][N]
};

// How the tiles of a grouped product are dealt to the eight XCDs (workgroup
// b runs on XCD b % 8; l = b / 8 counts an XCD's workgroups).  A band of
// column tiles of every row tile per XCD keeps the row tiles of one expert
// and column on one L2 -- but with few column tiles the bands are uneven (11
// column tiles: five XCDs get two columns, one gets one, two get none), so
// when more than a sixteenth of the band slots would be empty the tiles go
// round the XCDs one by one instead, row tile after row tile.
__device__ __forceinline__ void deal_grouped_tile(int n_tiles, int xcd, int l, int& tile_m, int& tile_n) {
  const int band = (n_tiles + 7) / 8;
  if ((band * 8 - n_tiles) * 16 > n_tiles) {
    const int g = l * 8 + xcd;
    tile_m = g / n_tiles;
    tile_n = g % n_tiles;
  } else {
    tile_m = l / band;
    tile_n = xcd * band + l % band;       // may be past the last column tile: the caller checks
  }
}

typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;

// fma(scale, q, bias) of small integer codes without converting them: a code in
// the low bits of a half word is the float16 denormal q * 2^-24 (a nibble
// further up q * 2^-20), v_fma_mix_f32 takes that as an operand, and with the
// scale times 2^24 (2^20) -- exact below kSmallScale -- it is the same product
// with the same one rounding, one instruction a code.  Eight four-bit codes take
// 17 vector instructions this way instead of 23, four eight-bit ones 9 instead of
// 10.
//
// A larger scale (float16 tables cannot hold one) becomes infinite, its weights
// infinite or NaN, and so every result of its column: the kernels look at one
// result a column when they are done and multiply such a column again
// (redo_column).  Over 160 products of 17 to 2048 rows that is 0.3 % in all; asked
// of the scales as they come by it was 1 %, up to 4 %.
constexpr float kSmallScale = 0x1p104f;

// Float16 weight tiles hold the weight times 2^6, which the results give back: then
// a weight of the smallest float16 scale, 2^-24, is off by 2^-7 of that at most --
// a bf16 tile's by up to 2^-9 of the weight, some eight scales -- and weights below
// 1023 fit.  (Scales of float16 weights lie around 2^-12 to 2^-4.)  A column with a
// larger one has no finite result and is multiplied again, plainly.
constexpr int kF16Shift = 6;
__device__ __forceinline__ u32x4 dequant_nibbles(uint32_t w, float s24, float s20, float bi) {
  const uint32_t w8 = w >> 8;
  const f16x2 a = __builtin_bit_cast(f16x2, w & 0x000F000Fu), b = __builtin_bit_cast(f16x2, w & 0x00F000F0u);
  const f16x2 c = __builtin_bit_cast(f16x2, w8 & 0x000F000Fu), d = __builtin_bit_cast(f16x2, w8 & 0x00F000F0u);
  const float f0 = fmaf((float)a[0], s24, bi), f4 = fmaf((float)a[1], s24, bi);
  const float f1 = fmaf((float)b[0], s20, bi), f5 = fmaf((float)b[1], s20, bi);
  const float f2 = fmaf((float)c[0], s24, bi), f6 = fmaf((float)c[1], s24, bi);
  const float f3 = fmaf((float)d[0], s20, bi), f7 = fmaf((float)d[1], s20, bi);
  return u32x4{pack_bf16x2(f0, f1), pack_bf16x2(f2, f3), pack_bf16x2(f4, f5), pack_bf16x2(f6, f7)};
}
__device__ __forceinline__ u32x2 dequant_bytes(uint32_t w, float s24, float bi) {
  const f16x2 a = __builtin_bit_cast(f16x2, w & 0x00FF00FFu), b = __builtin_bit_cast(f16x2, (w >> 8) & 0x00FF00FFu);
  const float f0 = fmaf((float)a[0], s24, bi), f2 = fmaf((float)a[1], s24, bi);
  const float f1 = fmaf((float)b[0], s24, bi), f3 = fmaf((float)b[1], s24, bi);
  return u32x2{pack_bf16x2(f0, f1), pack_bf16x2(f2, f3)};
}

// The same to float16 weights (tables times 2^kF16Shift, s24 and s20 as above):
// v_fma_mixlo / mixhi round to float16 as they go, so that eight four-bit codes
// take 13 vector instructions, eight eight-bit ones 11.
__device__ __forceinline__ u32x4 dequant_nibbles_f16(uint32_t w, float s24, float s20, float bi) {
  const uint32_t w8 = w >> 8;
  const f16x2 a = __builtin_bit_cast(f16x2, w & 0x000F000Fu), b = __builtin_bit_cast(f16x2, w & 0x00F000F0u);
  const f16x2 c = __builtin_bit_cast(f16x2, w8 & 0x000F000Fu), d = __builtin_bit_cast(f16x2, w8 & 0x00F000F0u);
  const f16x2 p0 = {(_Float16)fmaf((float)a[0], s24, bi), (_Float16)fmaf((float)b[0], s20, bi)};
  const f16x2 p1 = {(_Float16)fmaf((float)c[0], s24, bi), (_Float16)fmaf((float)d[0], s20, bi)};
  const f16x2 p2 = {(_Float16)fmaf((float)a[1], s24, bi), (_Float16)fmaf((float)b[1], s20, bi)};
  const f16x2 p3 = {(_Float16)fmaf((float)c[1], s24, bi), (_Float16)fmaf((float)d[1], s20, bi)};
  return u32x4{__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1), __builtin_bit_cast(uint32_t, p2),
               __builtin_bit_cast(uint32_t, p3)};
}
__device__ __forceinline__ u32x2 dequant_bytes_f16(uint32_t w, float s24, float bi) {
  const f16x2 a = __builtin_bit_cast(f16x2, w & 0x00FF00FFu), b = __builtin_bit_cast(f16x2, (w >> 8) & 0x00FF00FFu);
  const f16x2 p0 = {(_Float16)fmaf((float)a[0], s24, bi), (_Float16)fmaf((float)b[0], s24, bi)};
  const f16x2 p1 = {(_Float16)fmaf((float)a[1], s24, bi), (_Float16)fmaf((float)b[1], s24, bi)};
  return u32x2{__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1)};
}

// 32 codes (one row, one 32-group) -> four 16-byte pieces of bf16 weights
template <int MODE, int BITS>
__device__ __forceinline__ u32x4 dequant_piece(const uint32_t* q, int pc, float sc, float bi) {
  if constexpr (MODE == 1) {
    // exact: the converter widens the two codes of a byte and applies the power-of-two scale
    const uint32_t w = q[pc];
    return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 0)),
                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 1)),
                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 2)),
                 __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, sc, 3))};
  } else if constexpr (BITS == 8) {
    const u32x2 lo = dequant_bytes(q[2 * pc], sc * 0x1p24f, bi), hi = dequant_bytes(q[2 * pc + 1], sc * 0x1p24f, bi);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  } else {
    return dequant_nibbles(q[pc], sc * 0x1p24f, sc * 0x1p20f, bi);
  }
}

// The weight row [n] of expert `e` as the long way reads it: without regard to time.
template <int BITS>
struct LongRow {
  const uint8_t* codes;
  const void *s, *b;
  int64_t entry;         // of the row's first group
  int tab, gshift;

  __device__ __forceinline__ LongRow(const uint32_t* w, const void* s_, const void* b_, int64_t e, int64_t n, int64_t N, int64_t K, int gshift_, int tab_)
      : codes(reinterpret_cast<const uint8_t*>(w) + (e * N + n) * (K * BITS / 8)), s(s_), b(b_), entry((e * N + n) * (K >> gshift_)), tab(tab_),
        gshift(gshift_) {}
  // Has it a scale that is not small in [k0, k1)?  (Eight at a time: rows of NaN lead here too.)
  __device__ __forceinline__ bool large(int k0, int k1) const {
    const int last = (k1 - 1) >> gshift;
    bool l = false;
#pragma nounroll
    for (int g = k0 >> gshift; g <= last; g += 8)
#pragma unroll
      for (int i = 0; i < 8; ++i) l |= !(fabsf(load_table_rt(s, entry + (g + i < last ? g + i : last), tab)) < kSmallScale);
    return l;
  }
  // ... or a weight that is no finite float16 once it is shifted, whatever its code?
  __device__ __forceinline__ bool large_f16(int k0, int k1) const {
    const int last = (k1 - 1) >> gshift;
    bool l = false;
#pragma nounroll
    for (int g = k0 >> gshift; g <= last; ++g) {
      const float sc = load_table_rt(s, entry + g, tab), bi = load_table_rt(b, entry + g, tab);
      l |= !(fmaxf(fabsf(bi), fabsf(fmaf(sc, (float)((1 << BITS) - 1), bi))) < 65504.f / (1 << kF16Shift));
    }
    return l;
  }
  __device__ __forceinline__ float unrounded(int k) const {
    const uint32_t code = BITS == 8 ? codes[k] : (uint32_t)codes[k >> 1] >> (4 * (k & 1)) & 15u;
    const int64_t g = entry + (k >> gshift);
    return fmaf(load_table_rt(s, g, tab), (float)code, load_table_rt(b, g, tab));
  }
  __device__ __forceinline__ double weight(int k) const {             // the bf16 tile's
    return (double)bf16_bits_to_f32(f32_to_bf16_bits(unrounded(k)));
  }
};

// Column n of the `blocks` row ranges [lo[i], hi[i]) over [k0, k1) again if its scales
// ask for it (the prefill kernels: activations re-laid, results in y, or in a split's
// part).  The kernel's own stores have to have landed.
template <int BITS>
__device__ __forceinline__ void redo_column(const Gemm2Args& a, int e, int n, const int (&lo)[2], const int (&hi)[2], int blocks, int k0, int k1,
                                            int split) {
  if (n >= a.N) return;
  const LongRow<BITS> row(a.w, a.s, a.b, e, n, a.N, a.K, a.gs == 32 ? 5 : a.gs == 64 ? 6 : 7, a.tab);
  if (!row.large(k0, k1)) return;                // an activation, or a sum that is out of range
#pragma nounroll
  for (int i = 0; i < blocks; ++i) {
#pragma nounroll
    for (int m = i ? lo[1] : lo[0]; m < (i ? hi[1] : hi[0]); ++m) {
      double sum = 0.0;
#pragma nounroll
      for (int k = k0; k < k1; ++k)
        sum = fma((double)bf16_bits_to_f32(static_cast<const uint16_t*>(a.ax)[((int64_t)(k >> 3) * a.Rp + m) * 8 + (k & 7)]), row.weight(k), sum);
      if (a.splits > 1) a.part[((int64_t)split * a.R + m) * a.N + n] = (float)sum;
      else store_out(a.y, (a.out_idx ? (int64_t)a.out_idx[m] : (int64_t)m) * a.N + n, (float)sum, a.y_dtype);
    }
  }
}

}  // namespace g2
}  // namespace qmm
