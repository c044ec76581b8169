// Quantized matmul for short row groups on gfx950: products of seventeen to a
// few hundred rows, dense or per expert, whose time is the weight's stream and
// its dequantization rather than the matrix cores.
//
// What bounds it.  A tile of at most 64 rows does little matrix work per weight
// byte: each weight has to come in from HBM once and be dequantized once
// (float32 fma, one rounding to bf16: the tile semantics of the prefill
// kernels), and the chip only has the bandwidth and the vector ALU for that when
// every compute unit takes part.  The prefill kernels cut the output into
// 128-column tiles and walk K serially in each, so 4096 output columns keep 32
// of 256 compute units busy.  Here K is split as well: over the eight
// wavefronts of a workgroup, whose sums meet in LDS, and over `splits`
// workgroups, whose float32 sums meet in a second, small launch.
//
// A workgroup takes up to 64 rows x 128 columns over a run of K, 256 codes a
// step (eight-bit codes: 128 -- 128 bytes of every weight row, whole lines).  A
// step's packed weight, table entries and activations come in with
// direct-to-LDS loads into a ring of three to five stages, activations from
// their own rows (nothing is re-laid first); one barrier a step.  The eight
// wavefronts are two column halves times four quarters of the step's K, so an
// activation byte that has come in feeds 128 columns and the vector-memory path
// (64 bytes a clock a compute unit), LDS, the vector ALU and the matrix cores
// are all busy for about as long as HBM needs to deliver the weight.  (A first
// form, eight independent wavefronts of 64 columns with the activations of
// each fetched straight into registers, moved 24 KB of activations per 8 KB of
// weight through that path and sat in issue most of the time.)
//
// Measured, bf16 activations and four-bit codes in groups of 64, against the
// prefill kernel on whole K: 48 rows of 4096 x 14336 104 -> 19.5 us, 17 rows of
// 4096 x 4096 35 -> 11, 48 rows of 14336 x 4096 37 -> 19.9; float16 activations and
// tables, 77 rows of 4096 x 4096 46 -> 21 -> 13.5 without terms.  Of the 19.5 us about 8 are
// fixed (launch, first data, the sums' second launch; 10 before the sums were written
// through L2 and read once); a step takes 0.76 us and 0.14 more per row
// block, the vector ALU's instructions about half of it.
//
// The dequantized weight never goes through LDS: a lane reads the eight bytes
// that hold its codes of a step and widens them straight into the operand layout
// of v_mfma_f32_16x16x32_bf16 (the order of k inside an instruction is free as
// long as both operands agree: lane quarter kg takes codes 16 kg .. 16 kg + 15
// of its wavefront's 64, eight per instruction).  Row blocks of sixteen, one to
// four a tile, so that 17 or 48 rows are not padded to 64.
//
// float16 / float32 activations are exact sums of two / three bf16 terms; each
// term is a row block of its own on the same weight fragments and the terms'
// float32 sums are added in the epilogue, so the weight is still streamed once.
// float16 ones with float16 tables need no terms (short_terms).
#include <type_traits>
#include <utility>

#include "qmm_gemm2_common.hpp"
#include "qmm_gemv_common.hpp"

namespace qmm {

namespace {

typedef __attribute__((address_space(3))) void lds_void;

constexpr int kCols = 128;                       // weight rows (output columns) of a workgroup
constexpr int kWaves = 8;                        // two column halves x four quarters of a step's K
constexpr int kLine = 128;                       // bytes of a weight row in a step
constexpr int kStageW = kCols * kLine;           // 16 KB
constexpr int kTabWin = 8 * kCols * 4;           // a table window in LDS: eight entries' (or entry pairs') dwords of every column
constexpr int kTabs = 4 * kTabWin;               // ring of four

// All but the newest N vector-memory loads landed, every LDS read done (the
// next direct-to-LDS load may overwrite what was read); also a compiler barrier.
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | 0x0070);
  asm volatile("" ::: "memory");
}

// Direct-to-LDS load, 16 bytes a lane.  AUX = 2: non-temporal (the weight's own
// bytes, read once a launch; activations and table lines are read again).
template <int AUX>
__device__ __forceinline__ void dma16(__amdgpu_buffer_rsrc_t r, unsigned char* dst, uint32_t voff, uint32_t soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void*)dst, 16, voff, soff, 0, AUX);
}

struct ShortArgs {
  const void* x;                // bf16 rows [x_rows][K]; several terms: planes of R rows each
  const uint32_t* w;            // [E, N, K*bits/32]
  const void* s;                // [E, N, K/gs]
  const void* b;
  void* y;                      // [R, N]
  float* part;                  // [splits][R][N] when splits > 1
  const int32_t* row_offsets;   // [E+1] or null
  const int32_t* src_row;       // optional gather of x's rows
  const int32_t* out_idx;       // optional row scatter for y
  int R, N, K, E, x_rows;
  int gshift, y_dtype;          // log2(group size)
  int terms, blocks;            // a tile's row blocks = terms * blocks (<= MB)
  int m_tiles, n_tiles, splits;
  uint32_t m_magic, n_magic;    // ceil(2^32 / d): workgroup numbers are divided by m_tiles and n_tiles with them
  int steps;                    // of K
  int win_shift, tab_odd;       // log2(steps whose entries are sixteen bytes of a table row); rows may start inside a dword
};

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>)
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <int MODE, int BITS, int MB>
struct ShortShape {
  static constexpr int kStep = kLine * 8 / BITS;               // codes a step: 256 | 128
  static constexpr int kRowA = kStep * 2;                      // bytes of an activation row in a step
  static constexpr int kStageA = MB * 16 * kRowA;
  static constexpr int kStage = kStageW + kStageA;
  static constexpr int kFit = (163840 - kTabs) / kStage;
  static constexpr int kDepth = kFit < 5 ? kFit : 5;           // stages in the ring
  static constexpr int kSums = kWaves * 4 * MB * 4 * 64 * 4;   // the wavefronts' sums, after the run
  static constexpr int kLds = kDepth * kStage + kTabs > kSums ? kDepth * kStage + kTabs : kSums;
  static_assert(kDepth >= 3 && kLds <= 163840, "three stages fit");
};

// TAB: QMM_BF16, QMM_F16 or QMM_F32 tables (MXFP4: QMM_BF16, its scales are widened to that).
// HALF: float16 rows times float16 tables as they are, weights rounded to float16.
template <int MODE, int BITS, int TAB, int MB, bool HALF>
__global__ __launch_bounds__(64 * kWaves, 2) void short_kernel(ShortArgs a) {
  using S = ShortShape<MODE, BITS, MB>;
  static_assert(!HALF || (MODE == 0 && TAB == QMM_F16), "float16 weights come from float16 tables");
  constexpr int D = S::kDepth;
  constexpr int SUB = S::kStep / 4;              // codes of a wavefront's quarter: 64 | 32
  constexpr int STEPS = SUB / 32;                // MFMA steps: 2 | 1
  constexpr int NAT = S::kStageA / 1024;         // activation loads a step
  constexpr int LA = (NAT + kWaves - 1) / kWaves;
  constexpr int LLO = 2 + NAT / kWaves;          // loads of a step and wavefront (the first half of them: one more where NAT is uneven)
  constexpr bool UNEVEN = NAT % kWaves != 0;
  static_assert(!UNEVEN || NAT % kWaves == kWaves / 2, "half of the wavefronts have one more");
  extern __shared__ __align__(16) unsigned char smem[];
  unsigned char* const tabs = smem + D * S::kStage;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 1, wk = wave >> 1;
  const int r16 = lane & 15, kg = lane >> 4;

  // ---- which tile?  Workgroup b runs on XCD b % 8.  An XCD takes a contiguous
  // run of (split, column tile, row tile), row tiles fastest: those share the
  // weight, and the column tiles of one split share its run of the activations.
  const uint32_t total = (uint32_t)(a.n_tiles * a.m_tiles * a.splits), per = (total + 7) / 8;
  const uint32_t l = blockIdx.x >> 3, t = (blockIdx.x & 7) * per + l;
  if (l >= per || t >= total) return;
  const uint32_t tq = a.m_tiles == 1 ? t : __umulhi(t, a.m_magic);
  const uint32_t tz = a.n_tiles == 1 ? tq : __umulhi(tq, a.n_magic);
  const int tile_m = (int)(t - tq * a.m_tiles), tile_n = (int)(tq - tz * a.n_tiles), z = (int)tz;
  const int tile_rows = a.blocks * 16;
  int e = 0, row_hi = a.R, m0 = tile_m * tile_rows;
  if (a.row_offsets) {
    const RowTile rt = find_row_tile(a.row_offsets, a.E, a.R, tile_rows, tile_m);
    if (!__builtin_amdgcn_readfirstlane(rt.found)) return;       // (a per-lane condition would make what follows per-lane too)
    e = rt.e; row_hi = rt.hi; m0 = rt.lo + rt.idx * tile_rows;
  }
  if (m0 >= row_hi) return;
  const int n0 = tile_n * kCols;
  const int sq = a.splits == 1 ? a.steps : a.steps / a.splits, sr = a.steps - sq * a.splits;
  const int s0 = z * sq + (z < sr ? z : sr), s1 = s0 + sq + (z < sr ? 1 : 0);

  constexpr int tabsz = MODE == 1 ? 1 : (TAB == QMM_F32 ? 4 : 2);
  const int ng = a.K >> a.gshift;
  const uint32_t pitch = (uint32_t)(a.K / 8) * BITS, tpitch = (uint32_t)(ng * tabsz);
  const int64_t wbytes = (int64_t)a.N * pitch;
  // (table sizes rounded up to whole dwords: a row may start or end in the middle of one)
  const int64_t tbytes = ((int64_t)a.N * tpitch + 3) / 4 * 4;
  const char* wp = reinterpret_cast<const char*>(a.w) + e * wbytes;
  const char* sp = static_cast<const char*>(a.s) + e * ((int64_t)a.N * tpitch);
  const char* bp = static_cast<const char*>(MODE == 1 ? a.s : a.b) + e * ((int64_t)a.N * tpitch);
  const int64_t xbytes = (int64_t)a.terms * a.x_rows * a.K * 2;

  // Line v of a column half in LDS holds weight row 4 (v % 16) + v / 16 of the
  // half, so that the four column blocks of a lane (lines 16 c + lane % 16) are
  // four neighbouring columns of the result.  Weight load q: lines 8 wave .. of
  // half q, piece p of line v at position p ^ ((v >> 1) & 7): the sixteen lines
  // that a quarter wavefront reads one piece of then fall on different banks.
  const int v8 = 8 * wave + (lane >> 3);
  const uint32_t gw = (uint32_t)((lane & 7) ^ ((v8 >> 1) & 7)) * 16;
  uint32_t wvo[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = n0 + 64 * q + 4 * (v8 & 15) + (v8 >> 4);
    wvo[q] = row < a.N ? (uint32_t)row * pitch + gw : kOutOfRange;
  }
  // Activation load q: 1 KB of the stage at 1024 (q * kWaves + wave): whole row
  // segments, piece p of row r at position p ^ (r & 15) of its low four bits.
  constexpr int PPR = S::kRowA / 16;             // pieces a row: 32 | 16
  uint32_t xvo[LA], xk;
#pragma unroll
  for (int q = 0; q < LA; ++q) {
    const int tr = (q * kWaves + wave) * (64 / PPR) + lane / PPR, lp = lane % PPR;        // row of the tile's blocks, position
    const uint32_t gp = (uint32_t)(lp ^ (tr & 15));
    const int blk = (q * kWaves + wave) * (64 / PPR) / 16;       // (uniform: a load stays inside a row block)
    const int term = (blk >= a.blocks ? 1 : 0) + (blk >= 2 * a.blocks ? 1 : 0);
    const int m = m0 + (blk - term * a.blocks) * 16 + (tr & 15);
    int src = -1;
    if (term < a.terms && m < row_hi) src = a.src_row ? a.src_row[m] : m;
    xk = gp * 8;                                 // (the same for every q: tr & 15 does not depend on it)
    xvo[q] = src >= 0 && src < a.x_rows ? (uint32_t)((term * a.x_rows + src) * a.K) * 2u + gp * 16 : kOutOfRange;
  }
  // ---- tables.  Sixteen bytes of a column's row hold the entries of `ws` steps
  // (a power of two).  Window i of the run is fetched by wavefronts 2 (i % 4) and
  // the next, a column a lane, into registers four steps before its first step,
  // and written to LDS two steps before, as dwords of (scale, bias) per entry --
  // two-byte tables; float32 ones: scale | bias planes; MXFP4: the scales of two
  // neighbouring blocks as bf16 -- so that a lane finds its four columns'
  // entries in one 16-byte read.
  const int win_shift = a.win_shift;             // log2(ws)
  const int tcol = 64 * (wave & 1) + lane;
  const uint32_t tvo = n0 + tcol < a.N ? (uint32_t)(n0 + tcol) * tpitch : kOutOfRange;
  const auto rs = make_rsrc(sp, tbytes);
  const auto rb = make_rsrc(bp, tbytes);
  u32x4 tw_s, tw_b;
  uint32_t tx_s = 0, tx_b = 0, tmis = 0;         // a row that starts inside a dword: one dword more, and how far in
  auto fetch_window = [&](int st) __attribute__((always_inline)) {      // the window that starts at step st
    const uint32_t at = tvo + (uint32_t)((st * S::kStep) >> a.gshift) * (uint32_t)tabsz, al = at & ~3u;
    tmis = at & 3u;
    tw_s = __builtin_amdgcn_raw_buffer_load_b128(rs, al, 0, 0);
    if constexpr (MODE == 0) tw_b = __builtin_amdgcn_raw_buffer_load_b128(rb, al, 0, 0);
    if (a.tab_odd) {
      tx_s = __builtin_amdgcn_raw_buffer_load_b32(rs, al + 16, 0, 0);
      if constexpr (MODE == 0) tx_b = __builtin_amdgcn_raw_buffer_load_b32(rb, al + 16, 0, 0);
    }
  };
  auto write_window = [&](int i) __attribute__((always_inline)) {       // window i of the run
    uint32_t* dst = reinterpret_cast<uint32_t*>(tabs + (i & 3) * kTabWin) + tcol;
    u32x4 vs = tw_s, vb = MODE == 0 ? tw_b : tw_s;
    if (a.tab_odd) {
      const uint32_t sh = tmis * 8;
      vs = u32x4{__builtin_amdgcn_alignbit(tw_s[1], tw_s[0], sh), __builtin_amdgcn_alignbit(tw_s[2], tw_s[1], sh),
                 __builtin_amdgcn_alignbit(tw_s[3], tw_s[2], sh), __builtin_amdgcn_alignbit(tx_s, tw_s[3], sh)};
      if constexpr (MODE == 0)
        vb = u32x4{__builtin_amdgcn_alignbit(tw_b[1], tw_b[0], sh), __builtin_amdgcn_alignbit(tw_b[2], tw_b[1], sh),
                   __builtin_amdgcn_alignbit(tw_b[3], tw_b[2], sh), __builtin_amdgcn_alignbit(tx_b, tw_b[3], sh)};
    }
    if constexpr (MODE == 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t e0 = (vs[j >> 1] >> (16 * (j & 1))) & 255u, e1 = (vs[j >> 1] >> (16 * (j & 1) + 8)) & 255u;
        dst[j * kCols] = (__float_as_uint(e8m0_to_f32(e0)) >> 16) | (__float_as_uint(e8m0_to_f32(e1)) & 0xFFFF0000u);
      }
    } else if constexpr (TAB == QMM_F32) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dst[j * kCols] = vs[j];
        dst[(4 + j) * kCols] = vb[j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        dst[(2 * j) * kCols] = byte_perm(vb[j], vs[j], 0x05040100u);
        dst[(2 * j + 1) * kCols] = byte_perm(vb[j], vs[j], 0x07060302u);
      }
    }
  };

  auto issue = [&](int st, int slot) __attribute__((always_inline)) {
    unsigned char* dst = smem + slot * S::kStage;
    const bool live = st < s1;                   // past the run: empty buffers, nothing is fetched and the counts stay
    const auto rw = make_rsrc(wp, live ? wbytes : 0);
    const auto rx = make_rsrc(a.x, live ? xbytes : 0);
    if ((st + 1) * S::kStep <= a.K || !live) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        // (several row tiles read the same weight: it stays in L2)
        if (a.m_tiles == 1) dma16<2>(rw, dst + (q * kWaves + wave) * 1024, wvo[q], (uint32_t)st * kLine);
        else dma16<0>(rw, dst + (q * kWaves + wave) * 1024, wvo[q], (uint32_t)st * kLine);
      }
#pragma unroll
      for (int q = 0; q < LA; ++q)
        if (NAT % kWaves == 0 || q * kWaves + wave < NAT)
          dma16<0>(rx, dst + kStageW + (q * kWaves + wave) * 1024, xvo[q], (uint32_t)st * S::kRowA);
    } else {                                     // a ragged last step: the pieces past K read as zeros
      const uint32_t wl = (uint32_t)st * kLine + gw < pitch ? 0u : kOutOfRange;
      const uint32_t xl = st * S::kStep + (int)xk < a.K ? 0u : kOutOfRange;
#pragma unroll
      for (int q = 0; q < 2; ++q) dma16<2>(rw, dst + (q * kWaves + wave) * 1024, wvo[q] | wl, (uint32_t)st * kLine);
#pragma unroll
      for (int q = 0; q < LA; ++q)
        if (NAT % kWaves == 0 || q * kWaves + wave < NAT)
          dma16<0>(rx, dst + kStageW + (q * kWaves + wave) * 1024, xvo[q] | xl, (uint32_t)st * S::kRowA);
    }
  };

  f32x4 acc[4][MB];
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[c][i] = f32x4{0.f, 0.f, 0.f, 0.f};

  // ---- where this lane's operands lie in a stage
  const uint32_t ao = (uint32_t)kStageW + (uint32_t)r16 * S::kRowA +
                      (((uint32_t)(BITS == 4 ? wk * 8 + kg * 2 : wk * 4 + kg) ^ (uint32_t)r16) << 4);
  const uint32_t wo = (uint32_t)(wn * 64 + r16) * kLine + (((uint32_t)(wk * 2 + (kg >> 1)) ^ (uint32_t)(r16 >> 1)) << 4) + (kg & 1) * 8;
  // entry (MXFP4: pair) of this lane's codes inside a step, and its four columns
  const int te = MODE == 1 ? wk : (wk * SUB + kg * (SUB / 4)) >> a.gshift;
  const uint32_t to = (uint32_t)(te * kCols + wn * 64 + 4 * r16) * 4;
  const uint32_t tstep = (uint32_t)(MODE == 1 ? 4 : S::kStep >> a.gshift) * kCols * 4;    // bytes of a step's entries in a window

  struct Ops {
    bf16x8 xa[STEPS][MB];
    u32x2 q[4];
    u32x4 t0, t1;
  };
  auto read_ops = [&](int st, int slot, Ops& o) __attribute__((always_inline)) {
    const unsigned char* base = smem + slot * S::kStage;
    const int i = st - s0;
    const unsigned char* tb = tabs + ((i >> win_shift) & 3) * kTabWin + (uint32_t)(i & ((1 << win_shift) - 1)) * tstep + to;
    o.t0 = *reinterpret_cast<const u32x4*>(tb);
    if constexpr (TAB == QMM_F32) o.t1 = *reinterpret_cast<const u32x4*>(tb + 4 * kCols * 4);
#pragma unroll
    for (int c = 0; c < 4; ++c) o.q[c] = *reinterpret_cast<const u32x2*>(base + wo + c * 16 * kLine);
#pragma unroll
    for (int j = 0; j < STEPS; ++j)
#pragma unroll
      for (int i2 = 0; i2 < MB; ++i2) o.xa[j][i2] = *reinterpret_cast<const bf16x8*>(base + (ao ^ (j * 16)) + i2 * 16 * S::kRowA);
  };
  // Weight fragment b = (column block b / STEPS, MFMA step b % STEPS), widened
  // while the matrix core works on the fragment before it.
  auto widen = [&](const Ops& o, auto bc) __attribute__((always_inline)) -> bf16x8 {
    constexpr int c = decltype(bc)::value / STEPS, j = decltype(bc)::value % STEPS;
    if constexpr (MODE == 1) {
      return widen_e2m1(o.q[c][j], __uint_as_float(kg >= 2 ? o.t0[c] & 0xFFFF0000u : o.t0[c] << 16));
    } else {
      float sc, bi;
      if constexpr (TAB == QMM_F32) {
        sc = __uint_as_float(o.t0[c]);
        bi = __uint_as_float(o.t1[c]);
      } else if constexpr (TAB == QMM_F16) {
        sc = f16_bits_to_f32(o.t0[c] & 0xFFFFu);
        bi = f16_bits_to_f32(o.t0[c] >> 16);
      } else {
        sc = __uint_as_float(o.t0[c] << 16);
        bi = __uint_as_float(o.t0[c] & 0xFFFF0000u);
      }
      const uint32_t q[2] = {o.q[c][BITS == 4 ? j : 0], o.q[c][1]};
      if constexpr (HALF) {
        const float s24 = sc * (float)(1 << (24 + g2::kF16Shift)), bs = bi * (float)(1 << g2::kF16Shift);
        if constexpr (BITS == 4) return __builtin_bit_cast(bf16x8, g2::dequant_nibbles_f16(q[0], s24, s24 * 0x1p-4f, bs));
        const u32x2 lo = g2::dequant_bytes_f16(q[0], s24, bs), hi = g2::dequant_bytes_f16(q[1], s24, bs);
        return __builtin_bit_cast(bf16x8, u32x4{lo[0], lo[1], hi[0], hi[1]});
      }
      return __builtin_bit_cast(bf16x8, g2::dequant_piece<0, BITS>(q, 0, sc, bi));
    }
  };
  auto math = [&](const Ops& o) __attribute__((always_inline)) {
    constexpr int NB = 4 * STEPS;
    bf16x8 wq = widen(o, std::integral_constant<int, 0>{});
    static_for<NB>([&](auto bc) __attribute__((always_inline)) {
      constexpr int b = decltype(bc)::value, c = b / STEPS, j = b % STEPS;
      bf16x8 wn8 = wq;
      if constexpr (b + 1 < NB) wn8 = widen(o, std::integral_constant<int, b + 1>{});
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        if constexpr (HALF)
          acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, o.xa[j][i]), __builtin_bit_cast(f16x8, wq), acc[c][i], 0, 0, 0);
        else
          acc[c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(o.xa[j][i], wq, acc[c][i], 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               // one MFMA,
        __builtin_amdgcn_sched_group_barrier(0x002, (20 + MB - 1) / MB, 0);   // a share of the next fragment's vector work
      }
      __builtin_amdgcn_sched_barrier(0);
      wq = wn8;
    });
  };
  // ---- the run.  Step i is multiplied out of registers while its successor's
  // operands are read from LDS, steps up to i + D - 1 are under way and i + D is
  // requested, into the slot of step i: every wavefront has it in registers when
  // it passes the barrier.
  const int duty = wave >> 1;
  auto window_at = [&](int st) {                 // the number of the window that starts at step st if it is this wavefront's, else -1
    const int i = st - s0, n = i >> win_shift;
    return st < s1 && (i & ((1 << win_shift) - 1)) == 0 && (n & 3) == duty ? n : -1;
  };
  {
    int mine = -1;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      if (window_at(s0 + d) >= 0) mine = d;      // (at most one: four windows are dealt over four pairs of wavefronts)
    if (mine >= 0) fetch_window(s0 + mine);
#pragma unroll
    for (int d = 0; d < D; ++d) issue(s0 + d, d);
    if (mine == 0 || mine == 1) write_window(window_at(s0 + mine));
  }
  if (UNEVEN && wave < kWaves / 2) wait_loads<(D - 1) * (LLO + 1)>();
  else wait_loads<(D - 1) * LLO>();
  __builtin_amdgcn_s_barrier();
  Ops even, odd;
  read_ops(s0, 0, even);
  int slot = 0;
  auto step = [&](int st, const Ops& cur, Ops& nxt) __attribute__((always_inline)) {
    if (UNEVEN && wave < kWaves / 2) wait_loads<(D - 2) * (LLO + 1)>();
    else wait_loads<(D - 2) * LLO>();
    __builtin_amdgcn_s_barrier();
    const int next = slot + 1 == D ? 0 : slot + 1;
    read_ops(st + 1, next, nxt);                 // (past the run: whatever the ring holds, never used)
    const int put = window_at(st + 2);
    if (put >= 0) write_window(put);
    if (window_at(st + 4) >= 0) fetch_window(st + 4);
    issue(st + D, slot);
    // (K is a multiple of 64: a quarter lies inside K or past it)
    if (st * S::kStep + wk * SUB < a.K) math(cur);
    slot = next;
  };
  for (int st = s0; st < s1; st += 2) {
    step(st, even, odd);
    if (st + 1 < s1) step(st + 1, odd, even);
  }
  wait_loads<0>();                               // nothing may still land in the ring: it becomes the summing area
  __syncthreads();

  // ---- the four quarters' sums meet in LDS, four columns of a row a lane; the
  // terms of a row are added up
  f32x4* sums = reinterpret_cast<f32x4*>(smem);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      sums[((wk * 2 + wn) * (MB * 4) + i * 4 + v) * 64 + lane] = f32x4{acc[0][i][v], acc[1][i][v], acc[2][i][v], acc[3][i][v]};
  __syncthreads();
  // wavefront (h = wn, v = wk) takes component v of every row block of half h
  f32x4* const own = sums + (wn * (MB * 4) + wk) * 64 + lane;           // ... and i * 4 * 64: nobody else reads them
  f32x4 r[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const f32x4* p = own + i * 4 * 64;
    r[i] = p[0];
#pragma unroll
    for (int k = 1; k < 4; ++k) r[i] += p[k * (2 * MB * 4 * 64)];
  }
  if constexpr (MB >= 2) {
    if (a.terms == 2) {
#pragma unroll
      for (int i = 0; i < MB / 2; ++i) r[i] += r[i + MB / 2];
    }
  }
  if constexpr (MB == 3) {
    if (a.terms == 3) r[0] += r[1] + r[2];
  }
  if constexpr (HALF) {
#pragma unroll
    for (int i = 0; i < MB; ++i) r[i] *= 1.f / (1 << g2::kF16Shift);
  }
  const int n = n0 + 64 * wn + 4 * r16;
  if constexpr (MODE == 0 && (TAB != QMM_F16 || HALF)) {
    // a scale too large for the short form of the dequantization: its column's results
    // are not finite, in rows of zeros either
    float probe = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) probe = fmaf(r[0][j], 0.f, probe);        // NaN if one is not
    if (__builtin_expect(__ballot(probe != probe) != 0ull, 0)) {
#pragma unroll
      for (int i = 0; i < MB; ++i) own[i * 4 * 64] = r[i];
      const int k0 = s0 * S::kStep, k1 = s1 * S::kStep < a.K ? s1 * S::kStep : a.K;
      // (a column with a finite result in any row has no such scale: it is an activation)
      uint32_t fin = 0;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (i < a.blocks && r[i][j] * 0.f == 0.f) fin |= 1u << j;
      fin |= __shfl_xor(fin, 16);
      fin |= __shfl_xor(fin, 32);
#pragma nounroll
      for (int j = 0; j < 4; ++j) {
        if (n + j >= a.N) break;
        if (fin >> j & 1) continue;
        const g2::LongRow<BITS> row(a.w, a.s, a.b, e, n + j, a.N, a.K, a.gshift, TAB);
        if (!(HALF ? row.large_f16(k0, k1) : row.large(k0, k1))) continue;       // an activation, or a sum that is out of range
#pragma nounroll
        for (int i = 0; i < a.blocks; ++i) {
          const int m = m0 + i * 16 + 4 * kg + wk;
          const int src = m >= row_hi ? -1 : a.src_row ? a.src_row[m] : m;
          double sum = 0.0;
          if (src >= 0 && src < a.x_rows)
#pragma nounroll
            for (int t = 0; t < a.terms; ++t)
#pragma nounroll
              for (int k = k0; k < k1; ++k) {
                const uint32_t x = static_cast<const uint16_t*>(a.x)[((int64_t)t * a.x_rows + src) * a.K + k];
                if constexpr (HALF) sum = fma((double)f16_bits_to_f32(x), (double)row.unrounded(k), sum);
                else sum = fma((double)bf16_bits_to_f32(x), row.weight(k), sum);
              }
          reinterpret_cast<float*>(own + i * 4 * 64)[j] = (float)sum;
        }
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) r[i] = own[i * 4 * 64];
    }
  }
  const bool v4 = (a.N & 3) == 0 && (a.splits > 1 || (reinterpret_cast<uintptr_t>(a.y) & 15u) == 0);
  // A split's sums are written through L2: left dirty there they are written back when the
  // kernel ends, ahead of the launch that adds them up (48 rows of 4096 x 14336 21.5 -> 20.7 us,
  // float16 77 of 4096 x 4096 14.5 -> 14.1; 6 and 5 MB of sums).
  const bool through = wide_sums(a.R, a.N);
  const auto rp = make_rsrc(a.part + (int64_t)z * a.R * a.N, through ? (int64_t)a.R * a.N * 4 : 0);
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int m = m0 + i * 16 + 4 * kg + wk;
    if (i >= a.blocks || m >= row_hi || n >= a.N) continue;
    const f32x4 v = r[i];
    if (a.splits > 1) {
      float* p = a.part + ((int64_t)z * a.R + m) * a.N + n;
      if (v4 && through) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rp, (uint32_t)(m * a.N + n) * 4u, 0, kWriteThrough);
      else if (v4) *reinterpret_cast<f32x4*>(p) = v;
      else
        for (int j = 0; j < 4; ++j) if (n + j < a.N) p[j] = v[j];
      continue;
    }
    const int64_t at = (a.out_idx ? (int64_t)a.out_idx[m] : (int64_t)m) * a.N + n;
    if (!v4) {
      for (int j = 0; j < 4; ++j) if (n + j < a.N) store_out(a.y, at + j, v[j], a.y_dtype);
    } else if (a.y_dtype == QMM_F32) {
      *reinterpret_cast<f32x4*>(static_cast<float*>(a.y) + at) = v;
    } else {
      u32x2 h;
      if (a.y_dtype == QMM_BF16) h = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      else h = u32x2{f32_to_f16_bits(v[0]) | (f32_to_f16_bits(v[1]) << 16), f32_to_f16_bits(v[2]) | (f32_to_f16_bits(v[3]) << 16)};
      *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(a.y) + at) = h;
    }
  }
}

// float16 / float32 activations as bf16 terms: plane t holds term t of every
// row (gathered through src_row when given).  Eight values a thread.
template <int TERMS, typename T>
__global__ __launch_bounds__(256) void short_terms_kernel(const T* __restrict__ x, const int32_t* __restrict__ src_row,
                                                          u32x4* __restrict__ out, int R, int x_rows, int K) {
  const int pieces = K / 8;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)R * pieces) return;
  const int row = (int)(i / pieces), piece = (int)(i - (int64_t)row * pieces);
  const int64_t src = src_row ? (int64_t)src_row[row] : (int64_t)row;
  float f[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) f[j] = 0.f;
  if (src >= 0 && src < x_rows) {                // an index outside x gathers a zero row
    if constexpr (sizeof(T) == 4) {
      const f32x4* p = reinterpret_cast<const f32x4*>(x + src * K) + piece * 2;
      const f32x4 v0 = p[0], v1 = p[1];
#pragma unroll
      for (int j = 0; j < 4; ++j) { f[j] = v0[j]; f[4 + j] = v1[j]; }
    } else {
      const u32x4 v = reinterpret_cast<const u32x4*>(x + src * K)[piece];
#pragma unroll
      for (int j = 0; j < 4; ++j) { f[2 * j] = f16_bits_to_f32(v[j] & 0xFFFFu); f[2 * j + 1] = f16_bits_to_f32(v[j] >> 16); }
    }
  }
#pragma unroll
  for (int t = 0; t < TERMS; ++t) {
    uint32_t h[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      uint32_t hi = __float_as_uint(f[j]) & 0xFFFF0000u;        // truncation: the remainder is exact
      if (f[j] != f[j]) hi |= 0x00400000u;                      // a NaN stays a NaN when its payload is cut
      h[j] = hi;
      f[j] = (hi & 0x7F800000u) == 0x7F800000u ? 0.f : f[j] - __uint_as_float(hi);   // inf / NaN stay in the first term
    }
    out[(int64_t)t * R * pieces + i] = u32x4{(h[0] >> 16) | h[1], (h[2] >> 16) | h[3], (h[4] >> 16) | h[5], (h[6] >> 16) | h[7]};
  }
}

struct ShortPlan { int mb, blocks, m_tiles, splits; double us; };

// Rows a tile: at most four row blocks of sixteen, terms included, dealt evenly.
// Splits: as many workgroups as make the product shortest.  `us` is that time,
// from a fit to products of 17 to 2048 rows, N and K 1024 to 14336: launch, a
// round of tiles over the compute units for every 256 workgroups, a step of 256
// four-bit (128 eight-bit) codes, the second launch and its traffic.  Checked
// against 228 dense products it is 5 % off on average; for groups, whose sizes
// differ, it comes out 11 to 19 % too short (profiles/prefill_plan_fits.txt).
ShortPlan short_plan(int64_t R, int64_t E, int64_t N, int64_t K, int bits, int mode, int terms, size_t part_bytes) {
  ShortPlan p;
  const int64_t most = terms == 1 ? 4 : terms == 2 ? 2 : 1;      // row blocks a tile can hold
  const int64_t avg = E > 1 ? ceil_div(R, E) : R;                // rows of a group
  if (E > 1) p.blocks = (int)ceil_div(avg * 3 / 2, (int64_t)16); // groups differ: room for half as many again
  else p.blocks = (int)ceil_div(ceil_div(R, ceil_div(R, most * 16)), (int64_t)16);
  if (p.blocks > most) p.blocks = (int)most;
  if (p.blocks < 1) p.blocks = 1;
  p.mb = p.blocks * terms;
  const int64_t rows = p.blocks * 16;
  // row tiles that exist (ragged groups that need several: three quarters of one more each)
  const int64_t live = E > 1 ? (avg * 3 / 2 <= rows ? E : (R + E * rows * 3 / 4) / rows) : ceil_div(R, rows);
  p.m_tiles = (int)(E > 1 ? ceil_div(R, rows) + E : ceil_div(R, rows));
  const int64_t nt = ceil_div(N, kCols), steps = ceil_div(K, bits == 8 ? 128 : 256);
  const char* env = experiment_env("QMM_SHORT_SPLITS");
  p.us = 1e30;
  p.splits = 1;
  double best = 1e30;
  for (int s = 1; s <= 16; s = s < 6 ? s + 1 : s < 8 ? 8 : s + 4) {
    if (s > 1 && (s > steps || (double)s * R * N * 4 > (double)part_bytes)) break;
    const int64_t wgs = live * nt * s;
    const double step = (bits == 8 ? 0.66 : mode == QMM_MODE_MXFP4 ? 0.88 : 1.0) * (0.76 + 0.14 * p.mb + 0.08 * (wgs < 256 ? wgs / 256.0 : 1.0));
    const double us = (mode == QMM_MODE_MXFP4 ? 2.4 : 3.4) + (terms > 1 ? 3.1 : 0.0) + (double)ceil_div(wgs, 256) * (3.4 + ceil_div(steps, s) * step) +
                      (s > 1 ? 2.3 + (double)s * R * N * 1.7e-6 : 0.0);
    double cost = us * (1.0 + 0.01 * s);         // (of two alike the one with fewer splits)
    if (env) cost = abs(s - atoi(env));
    if (cost < best) { best = cost; p.us = us; p.splits = s; }
  }
  return p;
}

template <int MODE, int BITS, int TAB, int MB, bool HALF>
void launch_mb(const ShortArgs& a, hipStream_t st) {
  constexpr size_t lds = ShortShape<MODE, BITS, MB>::kLds;
  constexpr auto kern = short_kernel<MODE, BITS, TAB, MB, HALF>;
  if (!lds_limit<kern, lds>()) return;
  const int64_t total = ceil_div((int64_t)a.n_tiles * a.m_tiles * a.splits, 8) * 8;
  hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(64 * kWaves), lds, st, a);
}

template <int MODE, int BITS, int TAB, bool HALF = false>
void launch_short(const ShortArgs& a, int mb, hipStream_t st) {
  if (mb == 1) launch_mb<MODE, BITS, TAB, 1, HALF>(a, st);
  else if (mb == 2) launch_mb<MODE, BITS, TAB, 2, HALF>(a, st);
  else if (mb == 3) launch_mb<MODE, BITS, TAB, 3, HALF>(a, st);
  else launch_mb<MODE, BITS, TAB, 4, HALF>(a, st);
}

template <int BITS>
void launch_affine(const ShortArgs& a, int tab, int mb, bool half, hipStream_t st) {
  if (half) launch_short<0, BITS, QMM_F16, true>(a, mb, st);
  else if (tab == QMM_BF16) launch_short<0, BITS, QMM_BF16>(a, mb, st);
  else if (tab == QMM_F16) launch_short<0, BITS, QMM_F16>(a, mb, st);
  else launch_short<0, BITS, QMM_F32>(a, mb, st);
}

}  // namespace

// Shapes the kernel can run: K a whole number of a wavefront's quarters, table
// rows whose windows hold what a step needs (float32 entries of groups of 32 do
// not fit sixteen bytes), 32-bit lane offsets.
bool short_supported(int64_t R, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab, int terms,
                     const void* s, const void* b) {
  if (K <= 0 || K % 64 || (mode == QMM_MODE_AFFINE && tab == QMM_F32 && gs == 32 && bits == 4)) return false;
  if ((reinterpret_cast<uintptr_t>(s) & 3u) || (mode == QMM_MODE_AFFINE && (reinterpret_cast<uintptr_t>(b) & 3u))) return false;
  const int64_t tabsz = mode == QMM_MODE_MXFP4 ? 1 : tab == QMM_F32 ? 4 : 2;
  if (E > 1 && (N * (K / gs) * tabsz) % 4) return false;         // an expert's tables start on a dword
  if (N * (K * bits / 8) >= (1ll << 31) || N * (K / gs) * 4 >= (1ll << 31)) return false;
  // (workgroup numbers are divided by multiplication: exact while number times divisor is below 2^32)
  const int64_t nt = ceil_div(N, kCols), mt = ceil_div(R, 16) + E;
  if (nt >= 4096 || mt >= 4096 || mt * nt * 16 >= (1 << 20)) return false;
  return terms * R * K < (1ll << 30);
}

// The terms that this kernel multiplies activations as: one for bf16, and for
// float16 ones whose tables are float16 too -- they go to the matrix cores as they
// are, with weights rounded to float16 (11 significant bits instead of the bf16
// tile's 8).  77 rows of 4096 x 4096 in groups of 128: 21.7 us
// in two terms (a launch for them, tiles of 32 rows), 14.8 like this (tiles of 48).
// (Groups of 32 keep the two terms and the bf16 tile.  Nothing in the kernel asks for
// that; what they would gain has not been measured.)
int short_terms(int x_dtype, int tab, int gs, int mode) {
  if (x_dtype == QMM_F16) return mode == QMM_MODE_AFFINE && tab == QMM_F16 && gs >= 64 ? 1 : 2;
  return x_dtype == QMM_F32 ? 3 : 1;
}

// The activations' terms (none where there is one), without the splits' sums.
size_t short_prep_bytes(int64_t R, int64_t K, int terms) {
  return terms == 1 ? 0 : ((size_t)terms * R * K * 2 + 255) / 256 * 256;
}

// ... and with the sums of as many splits as the dense product would take
size_t short_workspace_bytes(int64_t R, int64_t N, int64_t K, int bits, int mode, int terms) {
  const ShortPlan p = short_plan(R, 1, N, K, bits, mode, terms, ~(size_t)0);
  return short_prep_bytes(R, K, terms) + (p.splits > 1 ? (size_t)p.splits * R * N * 4 : 0);
}

// About how long the product takes, in microseconds.
double short_us(int64_t R, int64_t E, int64_t N, int64_t K, int bits, int mode, int terms, size_t part_bytes) {
  return short_plan(R, E, N, K, bits, mode, terms, part_bytes).us;
}

void short_geometry(int64_t R, int64_t N, int64_t K, int bits, int mode, int* grid) {
  const ShortPlan p = short_plan(R, 1, N, K, bits, mode, 1, ~(size_t)0);
  *grid = (int)(ceil_div(N, kCols) * p.m_tiles * p.splits);
}

// x [x_rows, K] (rows gathered through src_row when given) times w [E, N, K]:
// rows [row_offsets[e], row_offsets[e+1]) of the gathered rows use expert e.
void short_dispatch(const void* x, int x_dtype, const void* w, const void* s, const void* b, int tab, void* y,
                    int y_dtype, const int32_t* row_offsets, const int32_t* src_row, const int32_t* out_idx, int64_t R,
                    int64_t x_rows, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, void* workspace,
                    size_t workspace_bytes, hipStream_t st) {
  const int terms = short_terms(x_dtype, tab, gs, mode);
  const size_t prep = short_prep_bytes(R, K, terms);
  const ShortPlan p = short_plan(R, row_offsets ? E : 1, N, K, bits, mode, terms, workspace_bytes - prep);
  ShortArgs a;
  a.x = x;
  a.w = static_cast<const uint32_t*>(w);
  a.s = s; a.b = b; a.y = y;
  a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + prep);
  a.row_offsets = row_offsets; a.src_row = src_row; a.out_idx = out_idx;
  a.R = (int)R; a.N = (int)N; a.K = (int)K; a.E = (int)E; a.x_rows = (int)x_rows;
  a.gshift = gs == 32 ? 5 : gs == 64 ? 6 : 7;
  a.y_dtype = y_dtype;
  a.terms = terms; a.blocks = p.blocks; a.m_tiles = p.m_tiles; a.splits = p.splits;
  a.n_tiles = (int)ceil_div(N, kCols);
  a.m_magic = (uint32_t)ceil_div(1ll << 32, a.m_tiles);
  a.n_magic = (uint32_t)ceil_div(1ll << 32, a.n_tiles);
  const int64_t step = bits == 8 ? 128 : 256, entry = mode == QMM_MODE_MXFP4 ? 1 : tab == QMM_F32 ? 4 : 2;
  a.steps = (int)ceil_div(K, step);
  a.win_shift = 0;
  while ((step / gs * entry) << (a.win_shift + 1) <= 16) ++a.win_shift;
  a.tab_odd = ((K / gs) * entry) % 4 != 0 || (step / gs * entry) % 4 != 0;
  if (terms > 1) {
    const dim3 pg((unsigned)ceil_div(R * (K / 8), 256));
    u32x4* out = static_cast<u32x4*>(workspace);
    if (terms == 3) hipLaunchKernelGGL((short_terms_kernel<3, float>), pg, dim3(256), 0, st, static_cast<const float*>(x), src_row, out, (int)R, (int)x_rows, (int)K);
    else hipLaunchKernelGGL((short_terms_kernel<2, uint16_t>), pg, dim3(256), 0, st, static_cast<const uint16_t*>(x), src_row, out, (int)R, (int)x_rows, (int)K);
    a.x = workspace;
    a.src_row = nullptr;
    a.x_rows = (int)R;
  }
  if (mode == QMM_MODE_MXFP4) launch_short<1, 4, QMM_BF16>(a, p.mb, st);
  else if (bits == 4) launch_affine<4>(a, tab, p.mb, terms == 1 && x_dtype == QMM_F16, st);
  else launch_affine<8>(a, tab, p.mb, terms == 1 && x_dtype == QMM_F16, st);
  if (p.splits > 1) split_sum_dispatch(a.part, y, y_dtype, R, N, p.splits, row_offsets, E, out_idx, st);
}

}  // namespace qmm
