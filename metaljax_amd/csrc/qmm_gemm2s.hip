// Prefill-regime quantized matmul on gfx950 with the wavefronts' roles split:
// the grouped (per-expert) product that the reference hands to mx.gather_qmm
// (src/metaljax/moe.py:1283-1340) and the dense product of
// mx.quantized_matmul (src/metaljax/qmm.py:2491) at M > 16, with the
// dequantization semantics of src/metaljax/qmm.py:71-79 (w = scale * q + bias
// as one fma).
//
// Why a second kernel.  In the general kernel every wavefront both
// dequantizes and multiplies, and a single wavefront a SIMD issues one
// instruction per four clocks, of any kind: the dequantization of a K-tile
// (about 100 vector ALU instructions per thread, the LDS writes, the loads
// that feed them) stands in the way of its own MFMAs.  With short row groups
// that is most of the time (a K-tile of a 128-row tile took 0.78 us of which
// the MFMAs were a third).
//
// So the roles are split, as in the decode kernel.  A workgroup is eight
// wavefronts, two a SIMD:
//   * producers (wavefronts 4-7) load the packed words and the scale / bias
//     windows, dequantize a K-tile (float32 fma, one round-to-nearest-even
//     to bf16: the reference's tile, bit for bit) two K-tiles ahead of its use
//     and write it to LDS one K-tile ahead;
//   * consumers (wavefronts 0-3) load their activation fragments (the re-laid
//     ax[k/8][row] form of the general kernel), read the weight fragments of
//     K-tile t from LDS and issue the MFMAs.
// One workgroup barrier per K-tile publishes tile t+1 and frees the stage of
// tile t-1 (three stages).
//
// Tile: up to 256 rows x 128 columns, and the rows a tile really holds pick
// one of three loops.  Up to 128 rows: consumer w multiplies row block w
// (32 rows) with the whole weight tile.  Up to 160: rows 128..159 are a fifth
// block split by columns, consumer w multiplies it with column block w.  More:
// consumer w multiplies row blocks w and w + 4 (every weight fragment read
// from LDS then feeds two MFMAs).  Longer experts take several tiles.
#include <algorithm>
#include <type_traits>

#include "qmm_gemm2_common.hpp"

namespace qmm {

namespace {

using namespace g2;

constexpr int kS = 3;                 // LDS stages: K-tile t lives in stage t % 3
constexpr int kAR = 3;                // activation fragments: K-tile t lives in ring slot t % 3 (t % 2 on full tiles)

// Table rows staged in LDS (a row's scales / biases of the whole K when they
// fit 128 bytes): 128 + 16 bytes a row, so that eight rows fall on different banks.
constexpr int kTabRow = 144;
constexpr int kTabKind = BN * kTabRow;

// TLDS: a tile's table rows are fetched once, into LDS (each row's line comes
// in once instead of once per four K-tiles); otherwise 16-byte windows per
// four K-tiles in registers.
// TAB: the tables' type (MXFP4: QMM_BF16, unused).
template <int MODE, int BITS, int TAB, bool G64, bool TLDS>
__global__ __launch_bounds__(512) void gemm2s_kernel(Gemm2Args a) {
  static_assert(!G64 || MODE == 0, "one group a K-tile is an affine layout");
  constexpr int WBITS = (MODE == 1) ? 4 : BITS;
  constexpr int WPT = 32 * WBITS / 32;             // packed words per producer thread and K-tile: 4 | 8
  extern __shared__ __align__(16) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // ---- which tile?  The grid is provisioned for the worst raggedness and
  // only the row tiles that exist are dealt (deal_grouped_tile: a band of
  // column tiles of every expert per XCD, expert after expert, or one by one
  // round the XCDs when the bands would be uneven).
  const int n_tiles = (a.N + BN - 1) / BN;
  const int xcd = blockIdx.x & 7, l = blockIdx.x >> 3;
  int tile_m, tile_n;
  deal_grouped_tile(n_tiles, xcd, l, tile_m, tile_n);
  int e = 0, row_lo = 0, row_hi = a.R, mt_idx = 0, split = 0;
  if (!a.row_offsets) {
    // one expert of all rows: an eighth of the grid takes a contiguous run of
    // tiles (and the workgroups that share a tile's K come one K range after the
    // other).  Tiles of 128 rows: column tile fastest, so that its workgroups share
    // few activation rows.  Ten tiles of 256 at most, where the last row tile may be a short
    // one: row tile fastest, so that every eighth has its share of the short ones and
    // reads a weight once (us, column / row tile fastest: 1106 rows of 6240 x 7424
    // 105.5 / 98.8, eight-bit 380 of 14712 x 1344 27.0 / 25.0 and 563 of 4712 x 13952
    // 104.7 / 100.7, 669 of 13856 x 2176 61.1 / 58.7, whole tiles 2048 of 4096 x 4096
    // 65.2 / 64.8; of 128 rows 500 of 6144 x 4096 37.4 / 38.5, 256 of 9216 x 3072 28.1 / 28.7).
    // More row tiles than that are more activations than the L2 of an XCD keeps for the next
    // column tile: 2190 rows of 8070 x 3008 187.7 / 171.9, but 5033 of 3112 x 832 39.7 / 46.0, 8174
    // of 3552 x 3712 218 / 280, float32 rows in three terms, 2674 of 7600 x 6656, 927 / 1157
    // (4073 drawn products, 0.2 % from the better order's time on average, row tile fastest in all 1.9 %).
    const int m_tiles = (a.R + a.tile_rows - 1) / a.tile_rows;
    const int tiles = n_tiles * m_tiles, total = tiles * a.splits, per = (total + 7) / 8;
    const int t = xcd * per + l;
    if (l >= per || t >= total) return;
    split = t / tiles;
    const int i = t - split * tiles;
    const bool by_rows = a.tile_rows == 256 && m_tiles <= 10;
    tile_m = by_rows ? i % m_tiles : i / n_tiles;
    tile_n = by_rows ? i / m_tiles : i % n_tiles;
    mt_idx = tile_m;
  } else {
    if (tile_n >= n_tiles) return;
    const RowTile rt = find_row_tile(a.row_offsets, a.E, a.R, a.tile_rows, tile_m);
    if (!rt.found) return;
    e = rt.e; row_lo = rt.lo; row_hi = rt.hi; mt_idx = rt.idx;
  }
  const int m0 = row_lo + mt_idx * a.tile_rows;
  if (m0 >= row_hi) return;
  const int m_end = row_hi < m0 + a.tile_rows ? row_hi : m0 + a.tile_rows;
  const int n0 = tile_n * BN;
  // This workgroup's K-tiles: KT of them from kb on, a multiple of four (whole
  // quads); K-tile numbers below count from kb.
  const int KA = a.K / BK, quads = (KA + 3) / 4;
  const int kb = a.splits == 1 ? 0 : quads * split / a.splits * 4;
  const int ke = a.splits == 1 ? KA : quads * (split + 1) / a.splits * 4;
  const int KT = (ke < KA ? ke : KA) - kb;
  auto clampk = [&](int kt) { return kt < KT ? kt : KT - 1; };

  if (wave >= 4) {
    // ======================= producers: the weight tile ====================
    const int ptid = tid - 256;
    const int wrow = ptid >> 1, whalf = ptid & 1;  // weight row of the tile, 32-code half of its K-tile
    const int64_t wpr = (int64_t)a.K * WBITS / 32;
    const int gs = (MODE == 1) ? 32 : a.gs;
    const int64_t ng = a.K / gs;
    constexpr int tabsz = (MODE == 1) ? 1 : (TAB == QMM_F32 ? 4 : 2);     // E8M0 bytes | float32 | 16-bit
    const uint32_t* wb = a.w + (int64_t)e * a.N * wpr;
    const char* sb = static_cast<const char*>(a.s) + (int64_t)e * a.N * ng * tabsz;
    const char* bb = (MODE == 1) ? sb : static_cast<const char*>(a.b) + (int64_t)e * a.N * ng * tabsz;
    int64_t wn_row = n0 + wrow;
    if (wn_row >= a.N) wn_row = a.N - 1;           // rows past N are computed and never stored
    const auto rw = make_rsrc(wb, (int64_t)a.N * wpr * 4);
    const uint32_t wvo = (uint32_t)((wn_row * wpr + whalf * WPT) * 4);
    struct WRegs { uint32_t q[WPT]; };
    auto load_w = [&](int kt, WRegs& r) {
      const uint32_t so = (uint32_t)(kb + kt) * (BK * WBITS / 8);
#pragma unroll
      for (int j = 0; j < WPT; j += 4) {
        const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, wvo + j * 4, so, 0);
        r.q[j] = v[0]; r.q[j + 1] = v[1]; r.q[j + 2] = v[2]; r.q[j + 3] = v[3];
      }
    };
    // scale / bias window: the entries of four K-tiles of this thread's row
    // (at most 16 bytes a table), fetched once per four K-tiles.  Where rows may
    // start inside a dword (tab_odd) a dword more is fetched and the window is
    // shifted into place.
    struct TabWin { u32x4 s, b; };
    const int64_t tbytes = ((int64_t)a.N * ng * tabsz + 3) / 4 * 4;
    const auto rs = make_rsrc(sb, tbytes);
    const auto rb = make_rsrc(bb, tbytes);
    const uint32_t tvo = (uint32_t)(wn_row * ng * tabsz);
    const int gshift = gs == 32 ? 5 : (gs == 64 ? 6 : 7);
    struct RawWin { u32x4 s, b; uint32_t xs, xb, mis; } rawn;
    auto load_win = [&](int quad, RawWin& r) {
      const uint32_t so = (uint32_t)((((kb + quad * 4) * BK) >> gshift) * tabsz);
      const uint32_t at = tvo + so, al = at & ~3u;
      r.s = __builtin_amdgcn_raw_buffer_load_b128(rs, al, 0, 0);
      if constexpr (MODE == 0) r.b = __builtin_amdgcn_raw_buffer_load_b128(rb, al, 0, 0);
      if constexpr (tabsz < 4) {
        if (a.tab_odd) {
          r.mis = (at & 3u) * 8;
          r.xs = __builtin_amdgcn_raw_buffer_load_b32(rs, al + 16, 0, 0);
          if constexpr (MODE == 0) r.xb = __builtin_amdgcn_raw_buffer_load_b32(rb, al + 16, 0, 0);
        }
      }
    };
    auto settle_win = [&](const RawWin& r, TabWin& tw) {
      tw.s = r.s;
      if constexpr (MODE == 0) tw.b = r.b;
      if constexpr (tabsz < 4) {
        if (a.tab_odd) {
          tw.s = u32x4{__builtin_amdgcn_alignbit(r.s[1], r.s[0], r.mis), __builtin_amdgcn_alignbit(r.s[2], r.s[1], r.mis),
                       __builtin_amdgcn_alignbit(r.s[3], r.s[2], r.mis), __builtin_amdgcn_alignbit(r.xs, r.s[3], r.mis)};
          if constexpr (MODE == 0)
            tw.b = u32x4{__builtin_amdgcn_alignbit(r.b[1], r.b[0], r.mis), __builtin_amdgcn_alignbit(r.b[2], r.b[1], r.mis),
                         __builtin_amdgcn_alignbit(r.b[3], r.b[2], r.mis), __builtin_amdgcn_alignbit(r.xb, r.b[3], r.mis)};
        }
      }
    };
    uint32_t eidx[4];                              // entry of K-tile t' inside its window, for this thread's half
#pragma unroll
    for (int t = 0; t < 4; ++t) eidx[t] = (uint32_t)((t * BK + whalf * 32) >> gshift);
    auto widen = [&](uint32_t v) -> float {        // a 16-bit entry (in the low half)
      return TAB == QMM_F16 ? f16_bits_to_f32(v & 0xFFFFu) : __uint_as_float(v << 16);
    };
    auto pick = [&](const u32x4& w, uint32_t ei) -> float {
      const uint32_t byte = ei * (uint32_t)tabsz;
      const uint32_t d = byte >> 2;
      uint32_t v = w[0];
      v = d == 1 ? w[1] : v;
      v = d == 2 ? w[2] : v;
      v = d == 3 ? w[3] : v;
      if constexpr (tabsz == 4) return __uint_as_float(v);
      v >>= (byte & 3u) * 8u;
      if constexpr (MODE == 1) return e8m0_to_f32(v & 255u);
      return widen(v);
    };
    unsigned char* tabs = smem + kS * kStage + wrow * kTabRow;
    const uint32_t tmis = tvo & 3u;                // staged rows start on a dword as well
    auto entry = [&](int kt, auto tqc, const TabWin& tw, float& sc, float& bi) {
      constexpr int tq = decltype(tqc)::value;
      if constexpr (TLDS) {
        const unsigned char* p = tabs + tmis + (((kb + kt) * BK + whalf * 32) >> gshift) * tabsz;
        if constexpr (MODE == 1) {
          sc = e8m0_to_f32(*p);
          bi = 0.f;
        } else if constexpr (tabsz == 4) {
          sc = *reinterpret_cast<const float*>(p);
          bi = *reinterpret_cast<const float*>(p + kTabKind);
        } else {
          sc = widen(*reinterpret_cast<const uint16_t*>(p));
          bi = widen(*reinterpret_cast<const uint16_t*>(p + kTabKind));
        }
      } else if constexpr (G64) {                          // one group a K-tile: entry tq for every thread
        if constexpr (tabsz == 4) {
          sc = __uint_as_float(tw.s[tq]);
          bi = __uint_as_float(tw.b[tq]);
        } else {
          sc = widen((tq & 1) ? tw.s[tq >> 1] >> 16 : tw.s[tq >> 1]);
          bi = widen((tq & 1) ? tw.b[tq >> 1] >> 16 : tw.b[tq >> 1]);
        }
      } else {
        sc = pick(tw.s, eidx[tq]);
        bi = MODE == 1 ? 0.f : pick(tw.b, eidx[tq]);
      }
    };
    // Pipeline of a weight tile: its words are requested a quad at a time,
    // seven to ten K-tiles before it is published, it is dequantized into
    // registers two K-tiles before, and written to LDS at the start of the
    // step before (the write then has the whole step to finish before the
    // barrier that publishes it).
    auto dequant_tile = [&](u32x4 (&dst)[4], const WRegs& r, float sc, float bi) {
#pragma unroll
      for (int pc = 0; pc < 4; ++pc) dst[pc] = dequant_piece<MODE, BITS>(r.q, pc, sc, bi);
    };
    auto write_tile = [&](int stage, const u32x4 (&src)[4]) {
#pragma unroll
      for (int pc = 0; pc < 4; ++pc)
        *reinterpret_cast<u32x4*>(smem + stage * kStage + swz(wrow, whalf * 4 + pc)) = src[pc];
    };
    TabWin tw_cur, tw_nxt;
    // Words of K-tile t live in wr[t % 12].  They are requested a quad (four
    // K-tiles) at a time: the four 16-byte pieces that a thread needs for a
    // quad lie in one 128-byte line of its row (four-bit codes; two lines with
    // eight-bit codes), and asked for one K-tile at a time the line came in
    // four times, each time evicted again by the 36 KB a K-tile moves through
    // the 32 KB L1.
    WRegs wr[12];
    u32x4 pend[4];                                  // the dequantized tile that the next step writes
    auto load_quad = [&](int kt0, auto sc0) __attribute__((always_inline)) {
      constexpr int s0 = decltype(sc0)::value;      // ring slot of tile kt0
#pragma unroll
      for (int i = 0; i < 4; ++i) load_w(clampk(kt0 + i), wr[(s0 + i) % 12]);
    };
    if constexpr (TLDS) {
      // this thread's half (64 bytes) of its row's table, per kind; the other
      // half is its neighbour lane's, and a wavefront's LDS accesses stay in order
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t o = (uint32_t)(whalf * 64 + i * 16);
        *reinterpret_cast<u32x4*>(tabs + o) = __builtin_amdgcn_raw_buffer_load_b128(rs, (tvo & ~3u) + o, 0, 0);
        if constexpr (MODE == 0)
          *reinterpret_cast<u32x4*>(tabs + kTabKind + o) = __builtin_amdgcn_raw_buffer_load_b128(rb, (tvo & ~3u) + o, 0, 0);
      }
    } else {
      load_win(0, rawn);
      settle_win(rawn, tw_cur);
    }
    load_quad(0, std::integral_constant<int, 0>{});
    load_quad(4, std::integral_constant<int, 4>{});
    tw_nxt = tw_cur;
    {
      float sc, bi;
      entry(0, std::integral_constant<int, 0>{}, tw_cur, sc, bi);
      dequant_tile(pend, wr[0], sc, bi);
      write_tile(0, pend);
      entry(clampk(1), std::integral_constant<int, 1>{}, tw_cur, sc, bi);
      dequant_tile(pend, wr[1], sc, bi);
    }
    lds_barrier();                                  // tile 0 is published
    __builtin_amdgcn_sched_barrier(0);
    // step kt runs beside the consumers' K-tile kt: it publishes tile kt + 1 and
    // dequantizes tile kt + 2 (past the last tile: clamped repeats into stages
    // that nobody reads)
    auto pstep = [&](int kt, auto tc) __attribute__((always_inline)) {
      constexpr int t12 = decltype(tc)::value;      // kt % 12
      constexpr int t = t12 & 3;
      write_tile((kt + 1) % kS, pend);
      if constexpr (t == 0) {
        // the quad two ahead, into the slots of the quad before this one
        // (its last tile was dequantized three steps ago)
        load_quad(kt + 8, std::integral_constant<int, (t12 + 8) % 12>{});
        if constexpr (!TLDS) {
          const int q = (kt >> 2) + 1;              // next quad's windows (clamped at the end)
          load_win(q * 4 < KT ? q : (kt >> 2), rawn);
        }
      }
      if constexpr (!TLDS && t == 2) settle_win(rawn, tw_nxt);
      float sc, bi;
      entry(clampk(kt + 2), std::integral_constant<int, (t + 2) & 3>{}, t >= 2 ? tw_nxt : tw_cur, sc, bi);
      // the step's barrier as soon as the write has landed (the consumers reach
      // theirs before their last k-step); the next tile's arithmetic after it
      lds_barrier();
      __builtin_amdgcn_sched_barrier(0);
      dequant_tile(pend, wr[(t12 + 2) % 12], sc, bi);
      if (t == 3) tw_cur = tw_nxt;
      __builtin_amdgcn_sched_barrier(0);
    };
    int kt = 0;
    for (; kt + 12 <= KT; kt += 12) {
      pstep(kt, std::integral_constant<int, 0>{});
      pstep(kt + 1, std::integral_constant<int, 1>{});
      pstep(kt + 2, std::integral_constant<int, 2>{});
      pstep(kt + 3, std::integral_constant<int, 3>{});
      pstep(kt + 4, std::integral_constant<int, 4>{});
      pstep(kt + 5, std::integral_constant<int, 5>{});
      pstep(kt + 6, std::integral_constant<int, 6>{});
      pstep(kt + 7, std::integral_constant<int, 7>{});
      pstep(kt + 8, std::integral_constant<int, 8>{});
      pstep(kt + 9, std::integral_constant<int, 9>{});
      pstep(kt + 10, std::integral_constant<int, 10>{});
      pstep(kt + 11, std::integral_constant<int, 11>{});
    }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 0>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 1>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 2>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 3>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 4>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 5>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 6>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 7>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 8>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 9>{}); ++kt; }
    if (kt < KT) { pstep(kt, std::integral_constant<int, 10>{}); ++kt; }
    return;
  }

  // ========================= consumers: the MFMAs ==========================
  const int wm = wave;                             // row block, and column block of the fifth
  const int li = lane & 31, kh = lane >> 5;
  // How many rows the tile holds decides the loop, for the whole workgroup:
  //   0: up to 128, one row block a consumer;
  //   1: up to 160, plus a fifth block split by columns;
  //   2: up to 256, two row blocks a consumer (w and w + 4).
  const int path = m_end - m0 <= 128 ? 0 : (m_end - m0 <= 160 ? 1 : 2);
  const bool five = path == 1, two = path == 2;
  // lane (row li, k-half kh) of k-step ks reads ax[(kt*8 + ks*2 + kh) * Rp + row]
  const auto ra = make_rsrc(a.ax, (int64_t)(a.K / 8) * a.Rp * 16);
  const uint32_t avo = (uint32_t)((kh * a.Rp + m0 + wm * 32 + li) * 16);
  // the second block: the fifth block's rows, or row block w + 4
  const uint32_t avo1 = avo + (uint32_t)(five ? (4 - wm) * 512 : 128 * 16);
  typedef u32x4 AFrag[4][2];
  auto load_a_part = [&](int kt, AFrag& dst, int ks, auto nac) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)(((kb + kt) * 8 + ks * 2) * 16) * (uint32_t)a.Rp;
    dst[ks][0] = __builtin_amdgcn_raw_buffer_load_b128(ra, avo, so, 0);
    if constexpr (decltype(nac)::value == 2) dst[ks][1] = __builtin_amdgcn_raw_buffer_load_b128(ra, avo1, so, 0);
  };

  f32x16 acc[4], acc2[4];                           // acc2[0] doubles as the fifth block's accumulator
#pragma unroll
  for (int r = 0; r < 16; ++r) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[j][r] = 0.f;
      acc2[j][r] = 0.f;
    }
  }
  AFrag af[kAR];
  bf16x8 fb[2][4], fbx[2];                          // B fragments: k-step ks in set ks & 1
  auto read_b = [&](const unsigned char* pbase, int ks, int set, auto fc) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      fb[set][j] = *reinterpret_cast<const bf16x8*>(pbase + swz(j * 32 + li, ks * 2 + kh));
    if constexpr (decltype(fc)::value)
      fbx[set] = *reinterpret_cast<const bf16x8*>(pbase + swz(wm * 32 + li, ks * 2 + kh));
  };

  auto run = [&](auto pathc) __attribute__((always_inline)) {
    constexpr int PATH = decltype(pathc)::value;
    constexpr bool FIVE = PATH == 1, TWO = PATH == 2;
    // activation K-tiles in registers: three (two K-tiles ahead), or two on a
    // full tile, whose 128 accumulator registers leave room for no more
    constexpr int AR = TWO ? 2 : 3;
    const std::integral_constant<int, PATH == 0 ? 1 : 2> nac;
    const std::integral_constant<bool, FIVE> fc;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) load_a_part(0, af[0], ks, nac);
    if constexpr (AR == 3) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) load_a_part(clampk(1), af[1], ks, nac);
    }
    lds_barrier();                                  // tile 0 is published
    read_b(smem, 0, 0, fc);
    auto cstep = [&](int kt, auto tc, auto ac) __attribute__((always_inline)) {
      constexpr int t = decltype(tc)::value;        // kt % 3: the LDS stage
      constexpr int as = decltype(ac)::value;       // kt % AR: the activation slot
      const unsigned char* pb = smem + t * kStage;
      constexpr int nstage = (t + 1) % kS;
      const int ktn = clampk(kt + AR - 1);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        // the next k-step's fragments; in the last k-step those of the next
        // tile, which the barrier below has published (past the last tile: a
        // stage that nobody reads)
        if (ks < 3) read_b(pb, ks + 1, (ks + 1) & 1, fc);
        else read_b(smem + nstage * kStage, 0, 0, fc);
        load_a_part(ktn, af[(as + AR - 1) % AR], ks, nac);
        // the fragment read last feeds the first MFMA: one LDS wait a k-step
        if constexpr (FIVE)
          acc2[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[as][ks][1]),
                                                            fbx[ks & 1], acc2[0], 0, 0, 0);
        const bf16x8 fa = __builtin_bit_cast(bf16x8, af[as][ks][0]);
#pragma unroll
        for (int j = 3; j >= 0; --j)
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa, fb[ks & 1][j], acc[j], 0, 0, 0);
        if constexpr (TWO) {
          const bf16x8 fa1 = __builtin_bit_cast(bf16x8, af[as][ks][1]);
#pragma unroll
          for (int j = 3; j >= 0; --j)
            acc2[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa1, fb[ks & 1][j], acc2[j], 0, 0, 0);
        }
        // order inside the k-step: the next k-step's fragment reads first (their
        // latency hides under this k-step's MFMAs), the loads spread between the MFMAs
        constexpr int NM = TWO ? 8 : (FIVE ? 5 : 4);
        __builtin_amdgcn_sched_group_barrier(0x100, FIVE ? 5 : 4, 0);
#pragma unroll
        for (int m = 0; m < NM; ++m) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          if (m < (PATH == 0 ? 1 : 2)) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        // One barrier a K-tile, before its last k-step: tile kt + 1 is
        // published (its producers wrote it at the start of their step), and
        // the producers learn that tile kt - 1 is read (they reuse its stage
        // in their next step).  The last k-step then fetches the next tile's
        // first fragments under its own MFMAs.
        if (ks == 2) lds_barrier();
      }
    };
    using std::integral_constant;
    int kt = 0;
    if constexpr (AR == 3) {
      for (; kt + 3 <= KT; kt += 3) {
        cstep(kt, integral_constant<int, 0>{}, integral_constant<int, 0>{});
        cstep(kt + 1, integral_constant<int, 1>{}, integral_constant<int, 1>{});
        cstep(kt + 2, integral_constant<int, 2>{}, integral_constant<int, 2>{});
      }
      if (kt < KT) { cstep(kt, integral_constant<int, 0>{}, integral_constant<int, 0>{}); ++kt; }
      if (kt < KT) { cstep(kt, integral_constant<int, 1>{}, integral_constant<int, 1>{}); ++kt; }
    } else {
      for (; kt + 6 <= KT; kt += 6) {
        cstep(kt, integral_constant<int, 0>{}, integral_constant<int, 0>{});
        cstep(kt + 1, integral_constant<int, 1>{}, integral_constant<int, 1>{});
        cstep(kt + 2, integral_constant<int, 2>{}, integral_constant<int, 0>{});
        cstep(kt + 3, integral_constant<int, 0>{}, integral_constant<int, 1>{});
        cstep(kt + 4, integral_constant<int, 1>{}, integral_constant<int, 0>{});
        cstep(kt + 5, integral_constant<int, 2>{}, integral_constant<int, 1>{});
      }
      if (kt < KT) { cstep(kt, integral_constant<int, 0>{}, integral_constant<int, 0>{}); ++kt; }
      if (kt < KT) { cstep(kt, integral_constant<int, 1>{}, integral_constant<int, 1>{}); ++kt; }
      if (kt < KT) { cstep(kt, integral_constant<int, 2>{}, integral_constant<int, 0>{}); ++kt; }
      if (kt < KT) { cstep(kt, integral_constant<int, 0>{}, integral_constant<int, 1>{}); ++kt; }
      if (kt < KT) { cstep(kt, integral_constant<int, 1>{}, integral_constant<int, 0>{}); ++kt; }
    }
  };
  if (two) run(std::integral_constant<int, 2>{});
  else if (five) run(std::integral_constant<int, 1>{});
  else run(std::integral_constant<int, 0>{});

  // ---- epilogue.  D of a 32x32 tile: lane holds column lane % 32 and rows
  // (r & 3) + 8 * (r >> 2) + 4 * (lane >> 5), r = 0..15.  Block 0 is row block
  // w over all columns; block 1 the fifth block's column block w, or row
  // block w + 4 over all columns.
  const bool wide = a.y_dtype != QMM_F32 && (a.N & 7) == 0 && a.splits == 1 &&
                    (reinterpret_cast<uintptr_t>(a.y) & 15u) == 0;
  if (wide) {
    // 16-bit outputs: transpose each 32-row block through this wavefront's
    // share of LDS (free after the last barrier), store 16 bytes a lane
    uint16_t* o16 = reinterpret_cast<uint16_t*>(smem) + wave * (32 * BN);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (i == 1 && !five && !two) break;
      const int ncb = (i == 0 || two) ? 4 : 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= ncb) break;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int rl = (r & 3) + 8 * (r >> 2) + 4 * kh;
          const float v = i == 0 ? acc[j][r] : acc2[j][r];
          o16[rl * BN + j * 32 + li] =
              (uint16_t)(a.y_dtype == QMM_BF16 ? f32_to_bf16_bits(v) : f32_to_f16_bits(v));
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int ppr = ncb * 4;                      // 16-byte pieces per row
      for (int q = 0; q < (32 * ppr) / 64; ++q) {
        const int idx = q * 64 + lane, rl = idx / ppr, pc = idx % ppr;
        const int m = m0 + (i == 0 ? wm : (two ? wm + 4 : 4)) * 32 + rl;
        const int n = n0 + ((i == 0 || two) ? 0 : wm * 32) + pc * 8;
        if (m < m_end && n < a.N) {
          const int64_t orow = a.out_idx ? (int64_t)a.out_idx[m] : (int64_t)m;
          // (not kept in L2, where the activations are read again: us, 2048 x 4096 x 4096 eight-bit
          // 70.1 -> 68.6, 380 of 14712 x 1344 27.8 -> 26.6, 1024 rows over 8 experts of 14336 x 4096
          // no more than runs differ; written through L2 instead it is 2 % slower than plain)
          __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(o16 + rl * BN + pc * 8),
                                      reinterpret_cast<u32x4*>(static_cast<uint16_t*>(a.y) + orow * a.N + n));
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  } else if (a.splits > 1 && wide_sums(a.R, a.N)) {
    // a split's float32 sums: the same transposition, sixteen bytes a lane written through
    // L2 (four bytes a lane as the accumulators lie: 642 rows of 1096 x 12800 40.7 us against
    // 36.3, 600 of 2048 x 12800 50.5 / 46.8, 900 of 4096 x 8192 73.8 / 69.7, 667 of it x 8064 61.4 / 59.0)
    float* o32 = reinterpret_cast<float*>(smem) + wave * (32 * BN);
    const auto rp = make_rsrc(a.part + (int64_t)split * a.R * a.N, (int64_t)a.R * a.N * 4);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (i == 1 && !five && !two) break;
      const int ncb = (i == 0 || two) ? 4 : 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= ncb) break;
#pragma unroll
        for (int r = 0; r < 16; ++r) o32[((r & 3) + 8 * (r >> 2) + 4 * kh) * BN + j * 32 + li] = i == 0 ? acc[j][r] : acc2[j][r];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const int ppr = ncb * 8;                      // 16-byte pieces per row
      for (int q = 0; q < (32 * ppr) / 64; ++q) {
        const int idx = q * 64 + lane, rl = idx / ppr, pc = idx % ppr;
        const int m = m0 + (i == 0 ? wm : (two ? wm + 4 : 4)) * 32 + rl;
        const int n = n0 + ((i == 0 || two) ? 0 : wm * 32) + pc * 4;
        if (m < m_end && n < a.N)
          __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(o32 + rl * BN + pc * 4), rp, (uint32_t)(m * a.N + n) * 4u, 0,
                                                 kWriteThrough);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (i == 1 && !five && !two) break;
      const int ncb = (i == 0 || two) ? 4 : 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j >= ncb) break;
        const int n = n0 + ((i == 0 || two) ? j : wm) * 32 + li;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = m0 + (i == 0 ? wm : (two ? wm + 4 : 4)) * 32 + (r & 3) + 8 * (r >> 2) + 4 * kh;
          if (m < m_end && n < a.N) {
            if (a.splits > 1) {
              __hip_atomic_store(a.part + ((int64_t)split * a.R + m) * a.N + n, i == 0 ? acc[j][r] : acc2[j][r], __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);      // (written through L2 as well)
              continue;
            }
            const int64_t orow = a.out_idx ? (int64_t)a.out_idx[m] : (int64_t)m;
            store_out(a.y, orow * a.N + n, i == 0 ? acc[j][r] : acc2[j][r], a.y_dtype);
          }
        }
      }
    }
  }
  if constexpr (MODE == 0 && TAB != QMM_F16) {
    // a scale too large for the short form of the dequantization: its column's results are not finite
    float probe = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) probe = fmaf(acc[j][0], 0.f, probe);          // NaN if one is not
    if (__builtin_expect(__ballot(probe != probe && kh == 0 && m0 + wm * 32 < m_end) != 0ull, 0)) {
      __builtin_amdgcn_s_waitcnt(0);
      // this wavefront's rows, a half of every block a lane: block w, and w + 4 or the fifth
      int lo[2], hi[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        lo[i] = m0 + (i == 0 ? wm : two ? wm + 4 : 4) * 32 + 16 * kh;
        hi[i] = lo[i] + 16 < m_end ? lo[i] + 16 : m_end;
      }
      // (a column with a finite result in any row has no such scale: it is an activation)
      uint32_t fin = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (m0 + wm * 32 + (r & 3) + 8 * (r >> 2) + 4 * kh < m_end && acc[j][r] * 0.f == 0.f) fin |= 1u << j;
      fin |= __shfl_xor(fin, 32);
#pragma nounroll
      for (int j = 0; j < 4; ++j)
        if (!(fin >> j & 1))
          redo_column<BITS>(a, e, n0 + j * 32 + li, lo, hi, two || (five && j == wm) ? 2 : 1, kb * BK, (kb + KT) * BK, split);
    }
  }
}

template <int MODE, int BITS, int TAB, bool G64, bool TLDS>
void launch_k(const Gemm2Args& a, hipStream_t st) {
  const int64_t m_tiles = ceil_div(a.R, a.tile_rows) + a.E;    // provisioned: a tile never straddles an expert
  int64_t total = ceil_div(ceil_div(a.N, BN), 8) * 8 * m_tiles;
  if (!a.row_offsets) total = ceil_div(ceil_div(a.N, BN) * ceil_div(a.R, a.tile_rows) * a.splits, 8) * 8;
  // (a split's results leave as float32 sums, a whole K's as 16-bit ones)
  constexpr size_t need = (size_t)(kS * kStage) + (TLDS ? 2 * kTabKind : 0), epi = (size_t)4 * 32 * BN * 2;
  constexpr size_t whole = std::max(need, epi), split = std::max(need, 2 * epi);
  constexpr auto kern = gemm2s_kernel<MODE, BITS, TAB, G64, TLDS>;
  if (!lds_limit<kern, split>()) return;
  const size_t lds = a.splits > 1 ? split : whole;
  hipLaunchKernelGGL(kern, dim3((unsigned)total), dim3(512), lds, st, a);
}

template <int MODE, int BITS, int TAB, bool G64>
void launch_s(const Gemm2Args& a, hipStream_t st) {
  // a row's table of the whole K (and the up to three bytes a row may start into
  // its first dword) in one 128-byte line per kind?
  const int64_t row_bytes = (MODE == 1 ? a.K / 32 : (int64_t)(a.K / a.gs) * (TAB == QMM_F32 ? 4 : 2)) + (a.tab_odd ? 3 : 0);
  static const bool no_tlds = experiment_env("QMM_GEMM2S_NOTLDS") != nullptr;
  if (row_bytes <= 128 && !no_tlds) launch_k<MODE, BITS, TAB, G64, true>(a, st);
  else launch_k<MODE, BITS, TAB, G64, false>(a, st);
}

template <int BITS, int TAB>
void launch_a(const Gemm2Args& a, hipStream_t st) {
  if (a.gs == 64) launch_s<0, BITS, TAB, true>(a, st);
  else launch_s<0, BITS, TAB, false>(a, st);
}

template <int BITS>
void launch_b(const Gemm2Args& a, hipStream_t st) {
  if (a.tab == QMM_BF16) launch_a<BITS, QMM_BF16>(a, st);
  else if (a.tab == QMM_F16) launch_a<BITS, QMM_F16>(a, st);
  else launch_a<BITS, QMM_F32>(a, st);
}

}  // namespace

// Every product whose tables can be fetched as 16-byte windows (four K-tiles'
// entries of a row: not float32 ones of groups of 32) from dword-aligned tables;
// the rest stays on the general kernel.
bool gemm2s_wanted(const g2::Gemm2Args& a, int mode, int bits) {
  if (experiment_env("QMM_GEMM2S") && experiment_env("QMM_GEMM2S")[0] == '0') return false;
  return (a.row_offsets ? a.E > 0 : a.E == 1) && a.tab_ok &&
         (mode == QMM_MODE_MXFP4 || ((bits == 4 || bits == 8) && !(a.tab == QMM_F32 && a.gs == 32)));
}

// Rows a tile may hold and workgroups that share its K: those that make the
// product shortest.  Returns that time in microseconds, from a fit to dense
// products of 17 to 2048 rows, N and K 1024 to 14336: the launches, a round for
// every 256 tiles (one workgroup fills a compute unit), a K-tile of up to 128 or
// up to 256 rows, the re-laid activations, the result, and a split K's sums.
// Checked against 68 four-bit and 68 eight-bit products it is 5 and 9 % off on
// average; for groups it comes out 7 and 18 % too short (without the launches of a
// caller that clears the result; profiles/prefill_plan_fits.txt).  Several experts keep 256-row
// tiles (every expert in one, and the short loop where it fits) and their whole
// K; for the row groups of a single expert (`row_offsets` with E = 1) the caller
// passes no room for sums, so that they keep theirs.
double gemm2s_plan(int64_t R, int64_t E, int64_t N, int64_t K, size_t part_bytes, int* tile_rows, int* splits) {
  const char* er = experiment_env("QMM_G2S_ROWS");
  const char* es = experiment_env("QMM_G2S_SPLITS");
  const int64_t kt = ceil_div(K, BK), quads = ceil_div(kt, 4), nt = ceil_div(N, BN), group = E > 1 ? ceil_div(R, E) : R;
  const bool wide = wide_sums(R, N);
  double best = 1e30, least = 1e30;
  *tile_rows = 256;
  *splits = 1;
  for (int rows = E > 1 ? 256 : 128; rows <= 256; rows += 128) {
    // (ragged groups: a quarter more rows than their mean to be expected in one)
    const int64_t mt = E > 1 ? E * ceil_div(group * 5 / 4, rows) : ceil_div(R, rows);
    const bool half = rows == 128 || (E > 1 ? group * 5 / 4 : R) <= 128;
    for (int s = 1; s <= (E > 1 ? 1 : 12); s = s < 6 ? s + 1 : s < 8 ? 8 : s + 4) {
      if (s > 1 && (s > quads || (double)s * R * N * 4 > (double)part_bytes)) break;
      const int64_t tiles = nt * mt * s;
      const double step = (half ? 0.41 : 0.60) + 0.105 * (tiles < 256 ? tiles / 256.0 : 1.0);
      const double sums = (double)s * R * N;     // (past 64 MB they come back from memory)
      const double us = 5.9 + (double)ceil_div(tiles, 256) * (2.5 + (s == 1 ? kt : 4 * ceil_div(quads, s)) * step) +
                        (double)R * K * 0.54e-6 + (double)R * N * 0.5e-6 +
                        (s == 1 ? 0.0 : wide ? 4.0 + (sums + std::max(0.0, sums - (1 << 24))) * 0.7e-6 : 4.6 + sums * 1.4e-6);
      // (of two alike the one with fewer splits, and none that makes a second round of one: 698
      // rows of 5432 x 7424 in three parts, 387 tiles, 75.7 us, whole 70.9)
      double cost = us * (1.0 + 0.01 * s) * (wide && s > 1 && tiles > 256 && nt * mt <= 256 ? 1.08 : 1.0);
      if (er && E <= 1 && atoi(er) != rows) cost += 1e9;
      if (es && E <= 1 && atoi(es) != s) cost += 1e9;
      if (cost < best) { best = cost; least = us; *tile_rows = rows; *splits = s; }
    }
  }
  return least;
}

void gemm2s_launch(const g2::Gemm2Args& a, int mode, int bits, hipStream_t st) {
  if (mode == QMM_MODE_MXFP4) launch_s<1, 4, QMM_BF16, false>(a, st);
  else if (bits == 4) launch_b<4>(a, st);
  else launch_b<8>(a, st);
}

}  // namespace qmm
