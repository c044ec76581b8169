// The small tensor work round an expert dispatch's products on gfx950, a launch a
// stretch of it: the router (logits, top-k, routing weights) and what lies between
// and behind the per-expert products (biases gathered by expert, slices,
// activations, the routing-weighted sum over a token's experts).  Reference
// src/metaljax/moe.py:335-442 and :1425-1461 run the same as one array operation
// after another.
//
// What bounds it: nothing here is more than a few hundred thousand elements, so a
// launch is its fixed cost and a few dependent loads: a pair map of 6 x 1024 takes
// 5.4 us, the row program of 3 tokens over 1024 x 8 router weights 7 (both cold;
// an empty launch is 2.7).  As array operations a block of 3 tokens over 8 experts
// of 1024 x 1024 was some thirty launches with their host work and three round
// trips to the host, 430 us; as the row program, two products and two maps it was 45,
// with each product and its map one launch and all of them issued by one library call
// it is 25, the host's and the device's alike.  They stay ahead as blocks grow and the
// products take over (us, launches / array operations, 8 experts of 1024 x 1024, top 2: 256
// tokens 93 / 439, 2048 tokens 364 / 815; 32 experts of 2880 x 2880, top 4: 64 tokens 286 /
// 533, 2048 tokens 3476 / 4536).
//
// The kernels interpret a short program that the planner wrote once (a product's, the
// map's behind it): the same instruction for every lane, operands in LDS (column of a lane: its own, so that no
// barrier is needed between instructions), arithmetic in float32, one rounding to the
// value's element type an instruction -- what an array operation of that type does.
#include <algorithm>
#include <cstddef>
#include <cstring>

#include "../../include/qmm_hip.h"
#include "qmm_gemv_common.hpp"

namespace qmm {

int moe_fail(int code, const char* what);        // qmm_api.hip: sets qmm_last_error
int moe_launched(const char* what);
int64_t skinny2_max_segments(int64_t P, int64_t E);
int device_cus();
int pair_product_route(const void* x, int x_dtype, int64_t P, int64_t E, int64_t N, int64_t K, const void* s, int y_dtype, int* waves);

namespace {

__device__ __forceinline__ float round_to(float v, int el) {
  if (el == QMM_EL_BF16) return bf16_bits_to_f32(f32_to_bf16_bits(v));
  if (el == QMM_EL_F16) return f16_bits_to_f32(f32_to_f16_bits(v));
  return v;
}

__device__ __forceinline__ float either_nan(float a, float b, float v) { return a != a ? a : b != b ? b : v; }

__device__ __forceinline__ float apply(int op, float a, float b, float c) {
  switch (op) {
    case QMM_OP_ADD: return a + b;
    case QMM_OP_SUB: return a - b;
    case QMM_OP_MUL: return a * b;
    case QMM_OP_DIV: return __fdiv_rn(a, b);
    case QMM_OP_MAX: return either_nan(a, b, fmaxf(a, b));
    case QMM_OP_MIN: return either_nan(a, b, fminf(a, b));
    case QMM_OP_POW: return powf(a, b);
    case QMM_OP_ABS: return fabsf(a);
    case QMM_OP_NEG: return -a;
    case QMM_OP_EXP: return expf(a);
    case QMM_OP_LOG: return logf(a);
    case QMM_OP_LOGISTIC: return __fdiv_rn(1.f, 1.f + expf(-a));
    case QMM_OP_TANH: return tanhf(a);
    case QMM_OP_SQRT: return __fsqrt_rn(a);
    case QMM_OP_RSQRT: return __fdiv_rn(1.f, __fsqrt_rn(a));
    case QMM_OP_CEIL: return ceilf(a);
    case QMM_OP_FLOOR: return floorf(a);
    case QMM_OP_RINT: return rintf(a);
    case QMM_OP_SIGN: return a != a ? a : a > 0.f ? 1.f : a < 0.f ? -1.f : a;
    case QMM_OP_EQ: return a == b ? 1.f : 0.f;
    case QMM_OP_NE: return a != b ? 1.f : 0.f;
    case QMM_OP_LT: return a < b ? 1.f : 0.f;
    case QMM_OP_LE: return a <= b ? 1.f : 0.f;
    case QMM_OP_GT: return a > b ? 1.f : 0.f;
    case QMM_OP_GE: return a >= b ? 1.f : 0.f;
    case QMM_OP_AND: return a != 0.f && b != 0.f ? 1.f : 0.f;
    case QMM_OP_OR: return a != 0.f || b != 0.f ? 1.f : 0.f;
    case QMM_OP_XOR: return (a != 0.f) != (b != 0.f) ? 1.f : 0.f;
    case QMM_OP_NOT: return a != 0.f ? 0.f : 1.f;
    case QMM_OP_SELECT: return a != 0.f ? b : c;
    case QMM_OP_CLAMP: {                           // min(max(b, low a), high c), NaN passed on
      const float m = either_nan(b, a, fmaxf(b, a));
      return either_nan(m, c, fminf(m, c));
    }
    default: return a;                             // QMM_OP_COPY
  }
}

// The dword that holds element i, shifted down to it: the same load whatever the
// type, so that several can be under way (with a branch on the type round each load
// they came one after the other).  The dword lies in the allocation that holds the
// element: those are whole dwords.
struct Raw { uint32_t word; uint32_t shift; };
__device__ __forceinline__ Raw load_raw(const void* p, int64_t i, int el) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(p) + (uint64_t)i * (el == QMM_EL_F32 ? 4u : el == QMM_EL_BOOL ? 1u : 2u);
  return Raw{*reinterpret_cast<const uint32_t*>(at & ~(uintptr_t)3), (uint32_t)(at & 3u) * 8u};
}
__device__ __forceinline__ float widen_raw(const Raw& r, int el) {
  if (el == QMM_EL_F32) return __uint_as_float(r.word);
  const uint32_t v = r.word >> r.shift;
  if (el == QMM_EL_BF16) return __uint_as_float(v << 16);
  if (el == QMM_EL_F16) return f16_bits_to_f32(v & 0xFFFFu);
  return (v & 0xFFu) ? 1.f : 0.f;
}
__device__ __forceinline__ void store_el(void* p, int64_t i, float v, int el) {
  if (el == QMM_EL_F32) static_cast<float*>(p)[i] = v;
  else if (el == QMM_EL_I32) static_cast<int32_t*>(p)[i] = (int32_t)v;
  else if (el == QMM_EL_BF16) static_cast<uint16_t*>(p)[i] = (uint16_t)f32_to_bf16_bits(v);
  else static_cast<uint16_t*>(p)[i] = (uint16_t)f32_to_f16_bits(v);
}

// An instruction out of LDS, into scalar registers: it is the same for all lanes.
// (The program is copied there when the kernel starts, a word a lane.  Read from the
// kernel's arguments one instruction after the other, each was a round trip of its own.)
template <class T>
__device__ __forceinline__ T uniform(const T& in) {
  constexpr int n = sizeof(T) / 4;
  union { T t; int w[n]; } u;
  u.t = in;
#pragma unroll
  for (int i = 0; i < n; ++i) u.w[i] = __builtin_amdgcn_readfirstlane(u.w[i]);
  return u.t;
}

constexpr int kThreads = 256;
// The sum over a token's pairs reads an expert's weight for each of them, where sorted
// pairs share it: while that is no more than the last-level caches deliver in the time of
// the launch that it spares.
constexpr int64_t kSumBytes = 16 << 20;

// A pair map's program over a lane's column of the register file.
__device__ __forceinline__ void run_map(const qmm_instruction* code, int instructions, float* r) {
  for (int n = 0; n < instructions; ++n) {
    const qmm_instruction q = uniform(code[n]);
    const float v = q.op == QMM_OP_IMM ? q.imm : apply(q.op, r[q.a * kThreads], r[q.b * kThreads], r[q.c * kThreads]);
    r[q.dst * kThreads] = round_to(v, q.el);
  }
}

// One output element a thread: its leaves are requested together (one round trip
// for all of them), then the program runs over its column of the register file.
__global__ __launch_bounds__(kThreads) void pair_map_kernel(qmm_pair_map a) {
  extern __shared__ float regs[];
  float* const r = regs + threadIdx.x;
  qmm_map_leaf* const leaves = reinterpret_cast<qmm_map_leaf*>(regs + a.registers * kThreads);
  qmm_instruction* const code = reinterpret_cast<qmm_instruction*>(leaves + QMM_MAP_LEAVES);
  if ((int)threadIdx.x < a.instructions) code[threadIdx.x] = a.code[threadIdx.x];
  else if (threadIdx.x >= 64 && (int)threadIdx.x - 64 < a.leaves) leaves[threadIdx.x - 64] = a.leaf[threadIdx.x - 64];
  __syncthreads();
  const int i = (int)blockIdx.x * kThreads + (int)threadIdx.x;
  const int per = a.weights ? a.per_token : 1;
  const int64_t row = (int64_t)blockIdx.z * gridDim.y + blockIdx.y;         // of y: a pair, a token
  if (i >= (int)a.inner || row * per >= a.pairs) return;
  int c[3] = {0, 0, i};
  if (a.rank > 1) { c[1] = i / (int)a.dims[2]; c[2] = i - c[1] * (int)a.dims[2]; }
  if (a.rank > 2) { c[0] = c[1] / (int)a.dims[1]; c[1] -= c[0] * (int)a.dims[1]; }
  float total = 0.f;
  for (int k = 0; k < per; ++k) {
    const int p = (int)row * per + k, t = p / a.per_token;
    const int e0 = __builtin_amdgcn_readfirstlane(a.experts_of[p]);
    const int e = e0 < 0 ? 0 : e0 >= a.experts ? a.experts - 1 : e0;
    Raw raw[QMM_MAP_LEAVES];
    int el[QMM_MAP_LEAVES];
#pragma unroll
    for (int j = 0; j < QMM_MAP_LEAVES; ++j) {
      if (j < a.leaves) {
        const qmm_map_leaf l = uniform(leaves[j]);
        const int64_t at = l.base + (int64_t)p * l.pair + (int64_t)e * l.expert + (int64_t)t * l.token;
        raw[j] = load_raw(l.p, at + (int64_t)c[0] * l.coef[0] + (int64_t)c[1] * l.coef[1] + (int64_t)c[2] * l.coef[2], l.el);
        el[j] = l.el;
      }
    }
#pragma unroll
    for (int j = 0; j < QMM_MAP_LEAVES; ++j)
      if (j < a.leaves) r[j * kThreads] = widen_raw(raw[j], el[j]);
    run_map(code, a.instructions, r);
    const float v = r[a.result * kThreads];
    if (!a.weights) {
      store_el(a.y, row * a.inner + i, v, a.y_el);
      return;
    }
    total += round_to(v, a.sum_el) * widen_raw(load_raw(a.weights, p, a.weights_el), a.weights_el);
  }
  store_el(a.y, row * a.inner + i, total, a.y_el);
}

// A product of MXFP4 experts and the pair map behind it, one launch.  A workgroup takes
// sixteen output elements of a pair (sorted: of up to sixteen pairs of one expert; SUM: of a
// token, WAVES wavefronts a pair, THREADS at most) and multiplies the weight rows that these read: tile t's
// row r is column col_base[t] + col_step[t] * element of the product.  The multiplication
// is the general decode kernel's (gemv_mxfp4_kernel: the same operands, in as many
// wavefronts, and so the same sums in the same order: a change to either's loop is one to
// both); its sums meet in LDS, where the map finds them as leaves.
//
// What bounds it: one round trip after the other -- arguments, the pair's expert, the
// weight -- with the map's memory leaves requested ahead of the weight: 6 pairs over 8
// experts of 2048 x 1024 and a map of two columns 11.3 us, of 1024 x 1024 and the sum of
// a token's two pairs 7.8 (a kernel trace of float32 rows); as two launches each 8.0 + 5.2
// and 6.5 + 5.1, and the gaps between them.
template <int T, int WAVES, int TERMS, int THREADS>
__global__ __launch_bounds__(THREADS ? THREADS : kWave* WAVES) void pair_product_kernel(qmm_pair_product a) {
  constexpr bool SUM = THREADS > 0;
  constexpr int XW = TERMS == 3 ? 2 : 1;           // 16-byte pieces of eight activations
  constexpr int U = THREADS == 1024 ? 1 : 2;       // macro chunks of 128 k whose loads are under way together (as registers allow)
  extern __shared__ float smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slice = wave % WAVES, group = wave / WAVES;
  const int r = lane & 15, kg = lane >> 4;
  const int all = SUM ? a.map.per_token * WAVES : WAVES;
  float* const red = smem;                         // [TERMS][all][T][4][64]
  float* const regs = red + TERMS * all * T * 4 * kWave;
  qmm_instruction* const code = reinterpret_cast<qmm_instruction*>(regs + a.map.registers * kThreads);
  int* const taken = reinterpret_cast<int*>(code + QMM_MAP_CODE) + wave * 16;
  float* const addends = reinterpret_cast<float*>(reinterpret_cast<int*>(code + QMM_MAP_CODE) + 16 * 16);    // [2][256]
  if ((int)threadIdx.x < a.map.instructions) code[threadIdx.x] = a.map.code[threadIdx.x];

  // ---- the pairs of this workgroup and the expert of this wavefront's
  const int z = (int)blockIdx.y, last = a.map.experts - 1;
  auto expert_of = [&](int p) __attribute__((always_inline)) {
    const int e = a.map.experts_of[p];
    return e < 0 ? 0 : e > last ? last : e;
  };
  int rows = SUM ? a.map.per_token : 1;
  int64_t e;
  if (!SUM && a.sorted) {
    rows = take_segment<true>(a.map.experts_of, (int)a.map.pairs, a.map.experts, z, lane, taken, e);
    if (rows == 0) return;                         // uniform, before any barrier
  } else {
    e = __builtin_amdgcn_readfirstlane(expert_of(SUM ? z * a.map.per_token + group : z));
  }
  // row m of the workgroup is pair ...
  auto pair_of = [&](int m) __attribute__((always_inline)) { return SUM ? z * a.map.per_token + m : a.sorted ? taken[m] : z; };

  // ---- the element of this thread (the first 256) and what its map reads from memory
  const int em = (threadIdx.x & 255) >> 4, er = threadIdx.x & 15;
  const int inner = (int)a.map.inner, element = (int)blockIdx.x * 16 + er;
  const bool mine = threadIdx.x < 256 && em < rows && element < inner;
  const int ep = mine ? pair_of(em) : 0;
  Raw raw[QMM_MAP_LEAVES], weight{0u, 0u};
  if (mine) {
    const int ee = SUM ? expert_of(ep) : (int)e, et = ep / a.map.per_token;
#pragma unroll
    for (int j = 0; j < QMM_MAP_LEAVES; ++j) {
      if (j < a.map.leaves && a.map.leaf[j].p) {
        const qmm_map_leaf& l = a.map.leaf[j];
        raw[j] = load_raw(l.p, l.base + (int64_t)ep * l.pair + (int64_t)ee * l.expert + (int64_t)et * l.token + (int64_t)element * l.coef[2], l.el);
      }
    }
    if constexpr (SUM) weight = load_raw(a.map.weights, ep, a.map.weights_el);
  }

  // ---- the product
  const int64_t wpr = a.k / 8;
  const int nblk = (int)(a.k / 32), chunks = (nblk + 3) / 4;
  const int c0 = (int)((int64_t)chunks * slice / WAVES), c1 = (int)((int64_t)chunks * (slice + 1) / WAVES);
  const uint32_t* wrow[T];
  const uint8_t* srow[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    int i = (int)blockIdx.x * 16 + r;
    if (i >= inner) i = inner - 1;
    const int64_t n = e * a.n + a.col_base[t] + (int64_t)i * a.col_step[t];
    wrow[t] = static_cast<const uint32_t*>(a.w) + n * wpr;
    srow[t] = static_cast<const uint8_t*>(a.s) + n * nblk;
  }
  int64_t src = -1;
  if (SUM ? r == 0 : r < rows) src = pair_of(SUM ? group : r) / a.x_per;
  const bool xvalid = src >= 0 && src < a.x_rows;
  const uint16_t* xrow = static_cast<const uint16_t*>(a.x) + (xvalid ? src : 0) * a.k * XW;
  f32x4 acc[TERMS][T];
#pragma unroll
  for (int term = 0; term < TERMS; ++term)
#pragma unroll
    for (int t = 0; t < T; ++t) acc[term][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int cb = c0; cb < c1; cb += U) {
    u32x4 q[U][T];
    uint8_t sraw[U][T];
    u32x4 xr[U][4][XW];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int blk = (cb + u) * 4 + kg;
      const bool live = cb + u < c1 && blk < nblk;
      if (!live) blk = nblk - 1;
#pragma unroll
      for (int t = 0; t < T; ++t) {
        q[u][t] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wrow[t] + (int64_t)blk * 4));
        sraw[u][t] = srow[t][blk];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int h = 0; h < XW; ++h) {
          xr[u][j][h] = u32x4{0u, 0u, 0u, 0u};
          if (xvalid && live) xr[u][j][h] = *reinterpret_cast<const u32x4*>(xrow + ((int64_t)blk * 32 + j * 8) * XW + h * 8);
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      float sc[T];
#pragma unroll
      for (int t = 0; t < T; ++t) sc[t] = e8m0_to_f32(sraw[u][t]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x8 xa[TERMS];                          // (zero where not live)
        operand_terms<TERMS>(xr[u][j], xa);
#pragma unroll
        for (int t = 0; t < T; ++t) {
          const bf16x8 wq = widen_e2m1(q[u][t][j], sc[t]);
#pragma unroll
          for (int term = 0; term < TERMS; ++term)
            acc[term][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xa[term], wq, acc[term][t], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int term = 0; term < TERMS; ++term)
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) red[(((term * all + wave) * T + t) * 4 + i) * kWave + lane] = acc[term][t][i];
  __syncthreads();

  // ---- the map
  float* const file = regs + (threadIdx.x & 255);
  float v = 0.f;
  if (mine) {
#pragma unroll
    for (int j = 0; j < QMM_MAP_LEAVES; ++j)
      if (j < a.map.leaves && a.map.leaf[j].p) file[j * kThreads] = widen_raw(raw[j], a.map.leaf[j].el);
    // (SUM: a pair's row is the first of its wavefronts' sixteen)
    const int first = SUM ? em * WAVES : 0, l = SUM ? er : 16 * (em >> 2) + er, i = SUM ? 0 : em & 3;
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float total = 0.f;
#pragma unroll
      for (int term = TERMS - 1; term >= 0; --term) {            // smallest first, in pairs: as gemv_mxfp4_kernel
        float part[WAVES];
#pragma unroll
        for (int wv = 0; wv < WAVES; ++wv) part[wv] = red[(((term * all + first + wv) * T + t) * 4 + i) * kWave + l];
#pragma unroll
        for (int d = 1; d < WAVES; d *= 2)
#pragma unroll
          for (int wv = 0; wv < WAVES; wv += 2 * d) part[wv] += part[wv + d];
        total = term == TERMS - 1 ? part[0] : total + part[0];
      }
      file[a.col_leaf[t] * kThreads] = round_to(total, a.product_el);
    }
    run_map(code, a.map.instructions, file);
    v = file[a.map.result * kThreads];
    if constexpr (!SUM) store_el(a.map.y, (int64_t)ep * inner + element, v, a.map.y_el);
  }
  if constexpr (SUM) {
    if (mine) {
      addends[threadIdx.x] = round_to(v, a.map.sum_el);
      addends[256 + threadIdx.x] = widen_raw(weight, a.map.weights_el);
    }
    __syncthreads();
    if (threadIdx.x >= 16 || element >= inner) return;
    float total = 0.f;
    for (int k = 0; k < rows; ++k) total += addends[k * 16 + er] * addends[256 + k * 16 + er];
    store_el(a.map.y, (int64_t)z * inner + element, total, a.map.y_el);
  }
}

constexpr int kRowThreads = 1024;
constexpr int kLeafTurns = 4;                      // elements of a leaf a lane holds while they arrive: 256 a leaf
static_assert(QMM_ROW_CODE <= 64 && QMM_MAP_CODE <= kThreads, "a program is held (copied) an instruction a lane (a thread)");
static_assert(QMM_ROW_LEAVES <= kRowThreads / 64, "a leaf a wavefront");

__device__ __forceinline__ void wave_lds_fence() {          // one wavefront's LDS accesses, in the order written
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Kernel arguments from byte FROM to byte TO, brought in together: a line of them that is
// first asked for where it is used is a round trip there, one line after the other.
template <int FROM, int TO, class T>
__device__ __forceinline__ void touch_arguments(const T& a) {
  constexpr int n = (TO - FROM + 63) / 64;
  static_assert(TO <= (int)sizeof(T) && FROM % 4 == 0 && n <= 24, "a word of every 64 bytes");
  const int* p = reinterpret_cast<const int*>(&a) + FROM / 4;
  int any = 0;
#pragma unroll
  for (int i = 0; i < n; ++i) any |= p[16 * i];
  asm volatile("" ::"s"(any));
}

template <int EL>
__device__ __forceinline__ float load_as(const void* p, uint32_t bytes) {
  const char* at = static_cast<const char*>(p) + bytes;
  if constexpr (EL == QMM_EL_F32) return *reinterpret_cast<const float*>(at);
  const uint32_t v = *reinterpret_cast<const uint16_t*>(at);
  return EL == QMM_EL_BF16 ? __uint_as_float(v << 16) : f16_bits_to_f32(v);
}

// sum over k = first, first + shares, ... < dot_k of x[t][k] w[k][n], both of type EL and
// within 2^31 bytes of a token's row and of the weight (the host looks).
template <int EL>
__device__ __forceinline__ float dot_share(const qmm_row_program& a, int64_t t, int n, int first, int shift) {
  constexpr uint32_t size = EL == QMM_EL_F32 ? 4 : 2;
  constexpr int kTurn = 8;                         // operand pairs under way together
  const char* x = static_cast<const char*>(a.dot_x) + t * a.dot_x_t * size;
  const uint32_t xk = (uint32_t)a.dot_x_k * size, wk = (uint32_t)a.dot_w_k * size, shares = 1u << shift;
  uint32_t xo = (uint32_t)first * xk, wo = (uint32_t)n * (uint32_t)a.dot_w_n * size + (uint32_t)first * wk;
  const uint32_t dx = shares * xk, dw = shares * wk;
  int left = ((int)a.dot_k - first + (int)shares - 1) >> shift;
  float sum = 0.f, xs[kTurn], ws[kTurn];
  for (; left >= kTurn; left -= kTurn) {
#pragma unroll
    for (int j = 0; j < kTurn; ++j, xo += dx, wo += dw) {
      xs[j] = load_as<EL>(x, xo);
      ws[j] = load_as<EL>(a.dot_w, wo);
    }
#pragma unroll
    for (int j = 0; j < kTurn; ++j) sum = fmaf(xs[j], ws[j], sum);
  }
  if (left > 0) {
#pragma unroll
    for (int j = 0; j < kTurn; ++j) {              // (past the last: the last again, not added)
      xs[j] = load_as<EL>(x, xo);
      ws[j] = load_as<EL>(a.dot_w, wo);
      if (j + 1 < left) { xo += dx; wo += dw; }
    }
#pragma unroll
    for (int j = 0; j < kTurn; ++j)
      if (j < left) sum = fmaf(xs[j], ws[j], sum);
  }
  return sum;
}

// Which form of the product: the element type of both operands, or -1 (as written).
int dot_form(const qmm_row_program& a) {
  if (!a.dot_x || a.dot_x_el != a.dot_w_el || a.dot_k > (1 << 28) || a.dot_x_k < 0 || a.dot_w_k < 0 || a.dot_w_n < 0 ||
      a.dot_x_k > (1 << 28) || a.dot_w_k > (1 << 28) || a.dot_w_n > (1 << 28))
    return -1;
  return a.dot_k * a.dot_x_k < (1 << 28) && a.dot_k * a.dot_w_k + a.dot_n * a.dot_w_n < (1 << 28) ? a.dot_x_el : -1;
}

// Keys that compare as the floats do: equal zeros are equal, every NaN is the same and the least.
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t b = __float_as_uint(v + 0.f);
  return v != v ? 0u : (b >> 31) ? ~b : b | 0x80000000u;
}

// One workgroup a token.  All sixteen wavefronts add up the logits (a thread a
// column and a share of the contraction, neighbouring threads along the dimension
// that is contiguous), the first one runs the program: a register is a row of
// floats in LDS, a lane takes elements lane, lane + 64, ...
//
// What bounds it: one wavefront's chain of waits and, as nothing else runs on its
// SIMD, of single instructions.  3 tokens over 1024 x 8 router weights and seven
// instructions took 10.2 us from the first wavefront's start: the program and the
// leaves 1.1, the product's operands behind them 2.2, ten rounds of a barrier for its
// sums 0.9, the instructions 4.9 (the top-k 1.2, a sum over two elements through six
// exchanges 0.9, 0.4 for the least), the stores 0.7.  So everything that memory holds
// is requested at once, sums meet behind one barrier, lane q keeps instruction q in
// registers, a top-k compares integer keys out of a scalar register and a reduction
// exchanges among as many lanes as there are elements: 6.4 (the operands 1.5, their sums 1.2, the
// instructions 3.2), the block of such tokens with 1024 x 1024 experts 29.2 -> 25.2.
__global__ __launch_bounds__(kRowThreads) void row_program_kernel(qmm_row_program a, int form) {
  extern __shared__ float regs[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = blockIdx.x;
  touch_arguments<0, offsetof(qmm_row_program, code)>(a);
  constexpr int kWords = sizeof(qmm_row_instruction) / 4;
  int code[kWords];                                // (wavefront 0) lane q: instruction q
#pragma unroll
  for (int w = 0; w < kWords; ++w) code[w] = 0;
  if (wave == 0 && lane < a.instructions) {
#pragma unroll
    for (int w = 0; w < kWords; ++w) code[w] = reinterpret_cast<const int*>(a.code + lane)[w];
  }
  Raw leaf[kLeafTurns];
  const bool leaves = wave < a.leaves;             // (eight leaves at most, sixteen wavefronts)
  const qmm_row_leaf l = a.leaf[leaves ? wave : 0];
  if (leaves) {
#pragma unroll
    for (int i = 0; i < kLeafTurns; ++i)
      if (lane + 64 * i < l.n) leaf[i] = load_raw(l.p, l.base + t * l.token + (int64_t)(lane + 64 * i) * l.step, l.el);
  }
  float* const part = regs + a.reg_floats;
  if (a.dot_x) {
    const int cols = a.dot_cols, log = 31 - __builtin_clz(cols), shift = 10 - log, shares = 1 << shift;
    const bool along_k = a.dot_w_k == 1;
    const int n = along_k ? (int)threadIdx.x >> shift : (int)threadIdx.x & (cols - 1);
    const int s = along_k ? (int)threadIdx.x & (shares - 1) : (int)threadIdx.x >> log;
    float sum = 0.f;
    if (n < a.dot_n) {
      if (form == QMM_EL_F32) {
        sum = dot_share<QMM_EL_F32>(a, t, n, s, shift);
      } else if (form == QMM_EL_BF16) {
        sum = dot_share<QMM_EL_BF16>(a, t, n, s, shift);
      } else if (form == QMM_EL_F16) {
        sum = dot_share<QMM_EL_F16>(a, t, n, s, shift);
      } else {
        const int64_t x0 = t * a.dot_x_t, w0 = n * a.dot_w_n;
#pragma unroll 4
        for (int64_t k = s; k < a.dot_k; k += shares)
          sum = fmaf(widen_raw(load_raw(a.dot_x, x0 + k * a.dot_x_k, a.dot_x_el), a.dot_x_el),
                     widen_raw(load_raw(a.dot_w, w0 + k * a.dot_w_k, a.dot_w_el), a.dot_w_el), sum);
      }
    }
    part[s * cols + n] = sum;
  }
  if (leaves) {
#pragma unroll
    for (int i = 0; i < kLeafTurns; ++i)
      if (lane + 64 * i < l.n) regs[l.dst + lane + 64 * i] = widen_raw(leaf[i], l.el);
    for (int i = lane + 64 * kLeafTurns; i < l.n; i += 64)
      regs[l.dst + i] = widen_raw(load_raw(l.p, l.base + t * l.token + (int64_t)i * l.step, l.el), l.el);
  }
  __syncthreads();
  if (wave) return;
  if (a.dot_x) {
    // share s of column n is part[s * cols + n]: a lane adds up those that lie a multiple of
    // max(cols, 64) apart, in pairs, then (fewer than 64 columns) the lanes of a column meet
    const int cols = a.dot_cols, apart = cols > 64 ? cols : 64, count = kRowThreads / apart;
    for (int n = lane; n < apart; n += 64) {
      float v[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) v[j] = part[(j & (count - 1)) * apart + n];
#pragma unroll
      for (int h = 8; h > 0; h /= 2)
        if (h < count) {
#pragma unroll
          for (int j = 0; j < h; ++j) v[j] += v[j + h];
        }
      float sum = v[0];
      for (int d = 32; d >= cols; d /= 2) sum += __shfl_xor(sum, d, 64);
      if (n < a.dot_n) regs[a.dot_dst + n] = round_to(sum, a.dot_el);
    }
  }
  for (int q0 = 0; q0 < a.instructions; ++q0) {
    wave_lds_fence();
    union { qmm_row_instruction q; int w[kWords]; } u;
#pragma unroll
    for (int w = 0; w < kWords; ++w) u.w[w] = __builtin_amdgcn_readlane(code[w], q0);
    const qmm_row_instruction& q = u.q;
    if (q.op <= QMM_OP_IMM) {
      const int am = q.an == 1 ? 0 : -1, bm = q.bn == 1 ? 0 : -1, cm = q.cn == 1 ? 0 : -1;
      for (int i = lane; i < q.n; i += 64) {
        const float v = q.op == QMM_OP_IMM ? q.imm : apply(q.op, regs[q.a + (i & am)], regs[q.b + (i & bm)], regs[q.c + (i & cm)]);
        regs[q.dst + i] = round_to(v, q.el);
      }
    } else if (q.op <= QMM_OP_ROWMIN) {            // sum, rowmax, rowmin
      const bool add = q.op == QMM_OP_SUM, most = q.op == QMM_OP_ROWMAX;
      auto both = [&](float x, float y) __attribute__((always_inline)) {
        return add ? x + y : either_nan(x, y, most ? fmaxf(x, y) : fminf(x, y));
      };
      float v = add ? 0.f : most ? -INFINITY : INFINITY;
      for (int i = lane; i < q.an; i += 64) v = both(v, regs[q.a + i]);
      // (lanes past the last element hold what changes nothing: they are met only where elements are)
      int d = 32;
      while (d >= q.an && d > 0) d /= 2;
      for (; d > 0; d /= 2) v = both(v, __shfl_xor(v, d, 64));
      if (lane == 0) regs[q.dst] = round_to(v, q.el);
    } else if (q.op == QMM_OP_SLICE) {
      for (int i = lane; i < q.n; i += 64) regs[q.dst + i] = round_to(regs[q.a + q.b + i * q.c], q.el);
    } else {
      // top-k: an element's place is the number of those ahead of it -- larger, or equal (NaN last) and of a
      // smaller index; key j counts from the element's own key on for j below it, above that from j = it on
      for (int i0 = 0; i0 < q.an; i0 += 64) {
        const int i = i0 + lane;
        const float v = regs[q.a + (i < q.an ? i : 0)];
        const uint32_t key = order_key(v);
        uint32_t place = 0;
        for (int j0 = 0; j0 < q.an; j0 += 64) {
          const int last = q.an - j0 < 64 ? q.an - j0 : 64;
          uint32_t others = order_key(regs[q.a + j0 + (lane < last ? lane : 0)]);
          if (lane >= last) others = 0u;           // (ahead of nobody: their places are past i)
          for (int j4 = 0; j4 < last; j4 += 4) {
#pragma unroll
            for (int j = j4; j < j4 + 4; ++j)
              place += (uint32_t)__builtin_amdgcn_readlane(others, j) >= key + (j0 + j >= i ? 1u : 0u) ? 1u : 0u;
          }
        }
        if ((i < q.an) & ((int)place < q.n)) {
          regs[q.dst + place] = v;
          regs[q.c + place] = (float)i;
        }
      }
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int j = 0; j < QMM_ROW_OUTS; ++j) {
    if (j >= a.outs) break;
    const qmm_row_out o = a.out[j];
    const int sm = o.srcn == 1 ? 0 : -1;
    for (int i = lane; i < o.n; i += 64) store_el(o.p, t * o.n + i, regs[o.src + (i & sm)], o.el);
  }
}

bool float_el(int el) { return el == QMM_EL_F32 || el == QMM_EL_BF16 || el == QMM_EL_F16; }
bool map_op(int op) { return op >= QMM_OP_COPY && op <= QMM_OP_IMM; }

// Every index that the program holds is checked here: what the kernel computes from
// it then stays inside the register file; addresses are the caller's shapes.
int check_map(const qmm_pair_map* a, bool product) {
  if (a->pairs < 0 || a->inner < 0 || a->per_token < 1 || a->pairs % a->per_token || a->experts < 1 || a->rank < 1 || a->rank > 3)
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: shape");
  if (a->pairs == 0 || a->inner == 0) return QMM_OK;
  if (a->inner > INT32_MAX - kThreads) return moe_fail(QMM_ERR_BAD_SHAPE, "pair map: a larger result than a grid takes");
  int64_t n = 1;
  for (int i = 0; i < a->rank; ++i) {
    if (a->dims[2 - i] < 1) return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: dimensions");
    n *= a->dims[2 - i];
  }
  if (n != a->inner || !a->experts_of || !a->y || !float_el(a->y_el) || !float_el(a->sum_el) || (a->weights && !float_el(a->weights_el)) || a->pairs > INT32_MAX)
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: pointers or types");
  if (a->leaves < 0 || a->leaves > QMM_MAP_LEAVES || a->instructions < 0 || a->instructions > QMM_MAP_CODE ||
      a->registers < 1 || a->registers > QMM_MAP_REGISTERS || a->leaves > a->registers || a->result < 0 || a->result >= a->registers)
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: program size");
  for (int i = 0; i < a->leaves; ++i)
    if ((!a->leaf[i].p && !product) || a->leaf[i].el < 0 || a->leaf[i].el > QMM_EL_BOOL) return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: leaf");
  for (int i = 0; i < a->instructions; ++i) {
    const qmm_instruction& q = a->code[i];
    if (!map_op(q.op) || q.dst >= a->registers || q.a >= a->registers || q.b >= a->registers || q.c >= a->registers || !float_el(q.el))
      return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair map: instruction");
  }
  return QMM_OK;
}

constexpr size_t kProductLds = 64 << 10;           // what a launch gets without asking for more
size_t pair_product_lds(const qmm_pair_product& a, int waves) {
  const qmm_pair_map& m = a.map;
  const int terms = a.x_el == QMM_EL_F32 ? 3 : a.x_el == QMM_EL_F16 ? 2 : 1;
  return ((size_t)terms * (m.weights ? m.per_token * waves : waves) * a.tiles * 4 * kWave + (size_t)m.registers * kThreads + 16 * 16 + 2 * 256) * 4 +
         sizeof(m.code);
}

// Is the sum over a token's pairs better as part of the product, in `groups` workgroups of
// `all` wavefronts?  Each has its own chain of round trips, so a round of them costs 3 to 8
// us where the launch that is spared is 3: one round always pays (by 1.1 to 2.2), a second
// where its workgroups are short (bf16 rows, one term) or the launches it stands for many
// (three pairs a token and more; long rows of sorted pairs excepted), and for 16-bit rows
// where the product alone would read an expert for every pair as well (bf16: any number).
// us, one launch / two, 8 experts: float32 5 and 12 tokens of two pairs over 1024 x 1024 13.4 /
// 12.3, 19.4 / 12.2, 3 over 8192 x 1024 37.9 / 27.1, 4 of four pairs 9.7 / 14.8, 8 17.5 / 15.0, 8 of
// K = 256 10.8 / 13.3; bf16 12 of two pairs over 1024 x 1024 9.9 / 11.2, 20 of K = 256 10.3 / 9.6.
// (10781 drawn products, weights in the caches and not: 0.4 % from the better one's time
// on average; the fused launch wherever it fits 6.3 %.  Whole blocks of float32, 24 tokens
// over 16 experts of 768 x 512 44.6 -> 31.6, 40 of one pair over 8 of 1024 x 512 36.1 -> 28.0.)
bool sum_pays(const qmm_pair_product& a, int all, size_t lds, bool sorted, int64_t groups) {
  const int terms = a.x_el == QMM_EL_F32 ? 3 : a.x_el == QMM_EL_F16 ? 2 : 1;
  if (terms == 1 && !sorted) return true;
  // wavefronts a SIMD holds by the kernels' registers: of 512 threads (142, 104, 88), of 1024 (104, 86, 62)
  constexpr int kHeld[2][3] = {{5, 4, 3}, {8, 5, 4}};
  const int64_t held = std::min<int64_t>(kHeld[all > 8][terms - 1] * 4 / all, (160 << 10) / (int64_t)lds);
  int rounds = terms == 1 || (terms == 2 && !sorted) ? 2 : 1;
  if (a.map.per_token > 2 && (!sorted || a.k * terms <= 2048)) ++rounds;
  return groups <= rounds * held * device_cus();
}

template <int T, int WAVES, int TERMS>
void launch_pair_product(const qmm_pair_product& a, dim3 grid, size_t lds, hipStream_t st) {
  const int all = a.map.weights ? a.map.per_token * WAVES : WAVES;
  if constexpr (T == 1) {
    if (a.map.weights) {
      if (all <= 8) hipLaunchKernelGGL((pair_product_kernel<T, WAVES, TERMS, 512>), grid, dim3(kWave * all), lds, st, a);
      else hipLaunchKernelGGL((pair_product_kernel<T, WAVES, TERMS, 1024>), grid, dim3(kWave * all), lds, st, a);
      return;
    }
  }
  hipLaunchKernelGGL((pair_product_kernel<T, WAVES, TERMS, 0>), grid, dim3(kWave * all), lds, st, a);
}

template <int T, int WAVES>
void launch_pair_product(const qmm_pair_product& a, dim3 grid, size_t lds, hipStream_t st) {
  if (a.x_el == QMM_EL_F32) launch_pair_product<T, WAVES, 3>(a, grid, lds, st);
  else if (a.x_el == QMM_EL_F16) launch_pair_product<T, WAVES, 2>(a, grid, lds, st);
  else launch_pair_product<T, WAVES, 1>(a, grid, lds, st);
}

}  // namespace
}  // namespace qmm

using namespace qmm;

extern "C" {

int qmm_pair_map_run(const qmm_pair_map* a, void* stream) {
  if (!a) return moe_fail(QMM_ERR_BAD_ARGUMENT, "null program");
  const int rc = check_map(a, false);
  if (rc || a->pairs == 0 || a->inner == 0) return rc;
  const int64_t rows = a->weights ? a->pairs / a->per_token : a->pairs;
  // (a grid's second axis ends at 65535; with more rows than that the third takes part)
  const int64_t planes = ceil_div(rows, 65535);
  const dim3 grid((unsigned)ceil_div(a->inner, kThreads), (unsigned)ceil_div(rows, planes), (unsigned)planes);
  const size_t lds = (size_t)a->registers * kThreads * 4 + sizeof(a->code) + sizeof(a->leaf);
  hipLaunchKernelGGL(pair_map_kernel, grid, dim3(kThreads), lds, static_cast<hipStream_t>(stream), *a);
  return moe_launched("pair map launch");
}

int qmm_pair_product_run(const qmm_pair_product* a, void* stream) {
  if (!a) return moe_fail(QMM_ERR_BAD_ARGUMENT, "null program");
  const qmm_pair_map& m = a->map;
  const int rc = check_map(&m, true);
  if (rc || m.pairs == 0 || m.inner == 0) return rc;
  if (!a->x || !a->w || !a->s || !float_el(a->x_el) || !float_el(a->product_el) || a->x_rows < 0 || a->x_per < 1 || a->n < 1 || a->k < 1 || a->k % 32)
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair product: operands");
  if (a->tiles < 1 || a->tiles > 2) return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair product: tiles");
  uint32_t from_product = 0;
  for (int t = 0; t < a->tiles; ++t) {
    if (a->col_leaf[t] < 0 || a->col_leaf[t] >= m.leaves || a->col_base[t] < 0 || a->col_step[t] < 0 ||
        a->col_base[t] + (m.inner - 1) * (int64_t)a->col_step[t] >= a->n)
      return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair product: columns");
    from_product |= 1u << a->col_leaf[t];
  }
  for (int i = 0; i < m.leaves; ++i)
    if ((m.leaf[i].p == nullptr) != ((from_product >> i & 1) != 0)) return moe_fail(QMM_ERR_BAD_ARGUMENT, "pair product: leaf");
  if (m.rank != 1 || a->mode != QMM_MODE_MXFP4) return moe_fail(QMM_ERR_UNSUPPORTED, "pair product: a result of several axes a pair, or affine experts");
  int waves = 4;
  int route = pair_product_route(a->x, a->x_el, m.pairs, m.experts, a->n, a->k, a->s, a->product_el, &waves);
  waves = waves == 4 ? 4 : 8;                      // (what there are launches of)
  if (m.weights && (a->tiles > 1 || m.per_token * waves > 16 || (route == 2 && m.pairs * (a->n * a->k / 2) > kSumBytes))) route = 0;
  const size_t lds = pair_product_lds(*a, waves);
  if (m.weights && route && !sum_pays(*a, m.per_token * waves, lds, route == 2, m.pairs / m.per_token * ceil_div(m.inner, 16))) route = 0;
  if (!route || (reinterpret_cast<uintptr_t>(a->w) & 15u) || lds > kProductLds) return moe_fail(QMM_ERR_UNSUPPORTED, "pair product: two launches are better");
  const int64_t segments = m.weights ? m.pairs / m.per_token : route == 2 ? skinny2_max_segments(m.pairs, m.experts) : m.pairs;
  qmm_pair_product p = *a;
  p.sorted = route == 2;
  const dim3 grid((unsigned)ceil_div(m.inner, 16), (unsigned)segments);
  const hipStream_t st = static_cast<hipStream_t>(stream);
  if (a->tiles == 1 && waves == 4) launch_pair_product<1, 4>(p, grid, lds, st);
  else if (a->tiles == 1) launch_pair_product<1, 8>(p, grid, lds, st);
  else if (waves == 4) launch_pair_product<2, 4>(p, grid, lds, st);
  else launch_pair_product<2, 8>(p, grid, lds, st);
  return moe_launched("pair product launch");
}

int qmm_row_program_run(const qmm_row_program* a, void* stream) {
  if (!a) return moe_fail(QMM_ERR_BAD_ARGUMENT, "null program");
  if (a->tokens < 0 || a->tokens > (1 << 30) || a->reg_floats < 1 || a->reg_floats > QMM_ROW_FLOATS || a->leaves < 0 ||
      a->leaves > QMM_ROW_LEAVES || a->instructions < 0 || a->instructions > QMM_ROW_CODE || a->outs < 0 || a->outs > QMM_ROW_OUTS)
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "row program: size");
  if (a->tokens == 0) return QMM_OK;
  auto in = [&](int64_t at, int64_t n) { return at >= 0 && n >= 1 && at + n <= a->reg_floats; };
  if (a->dot_x && (!a->dot_w || a->dot_k < 1 || a->dot_n < 1 || a->dot_cols < a->dot_n || a->dot_cols > kRowThreads ||
                   (a->dot_cols & (a->dot_cols - 1)) || !in(a->dot_dst, a->dot_n) || !float_el(a->dot_x_el) ||
                   !float_el(a->dot_w_el) || !float_el(a->dot_el)))
    return moe_fail(QMM_ERR_BAD_ARGUMENT, "row program: product");
  for (int i = 0; i < a->leaves; ++i)
    if (!a->leaf[i].p || !in(a->leaf[i].dst, a->leaf[i].n) || a->leaf[i].el < 0 || a->leaf[i].el > QMM_EL_BOOL)
      return moe_fail(QMM_ERR_BAD_ARGUMENT, "row program: leaf");
  for (int i = 0; i < a->instructions; ++i) {
    const qmm_row_instruction& q = a->code[i];
    bool ok = float_el(q.el) && in(q.dst, q.op == QMM_OP_SUM || q.op == QMM_OP_ROWMAX || q.op == QMM_OP_ROWMIN ? 1 : q.n);
    if (q.op == QMM_OP_TOPK) ok = ok && in(q.a, q.an) && in(q.c, q.n) && q.n <= q.an;
    else if (q.op == QMM_OP_SUM || q.op == QMM_OP_ROWMAX || q.op == QMM_OP_ROWMIN) ok = ok && in(q.a, q.an);
    else if (q.op == QMM_OP_SLICE) ok = ok && in(q.a, q.an) && q.b >= 0 && q.c >= 1 && q.b + (int64_t)(q.n - 1) * q.c < q.an;
    else if (q.op != QMM_OP_IMM)
      ok = ok && map_op(q.op) && in(q.a, q.an) && in(q.b, q.bn) && in(q.c, q.cn) && (q.an == 1 || q.an >= q.n) &&
           (q.bn == 1 || q.bn >= q.n) && (q.cn == 1 || q.cn >= q.n);
    if (!ok) return moe_fail(QMM_ERR_BAD_ARGUMENT, "row program: instruction");
  }
  for (int i = 0; i < a->outs; ++i)
    if (!a->out[i].p || a->out[i].n < 1 || !in(a->out[i].src, a->out[i].srcn) || (a->out[i].srcn != 1 && a->out[i].srcn < a->out[i].n) ||
        !(float_el(a->out[i].el) || a->out[i].el == QMM_EL_I32))
      return moe_fail(QMM_ERR_BAD_ARGUMENT, "row program: output");
  const size_t lds = ((size_t)a->reg_floats + (a->dot_x ? kRowThreads : 0)) * 4;
  hipLaunchKernelGGL(row_program_kernel, dim3((unsigned)a->tokens), dim3(kRowThreads), lds, static_cast<hipStream_t>(stream), *a, dot_form(*a));
  return moe_launched("row program launch");
}

int qmm_steps_run(const qmm_step* steps, int64_t n, const uint64_t* values, int64_t n_values, void* stream) {
  if (n < 0 || (n && !steps) || (n_values && !values)) return moe_fail(QMM_ERR_BAD_ARGUMENT, "null steps");
  union { qmm_row_program rows; qmm_pair_product product; qmm_pair_map map; qmm_pair_gather gather; } u;
  constexpr size_t sizes[] = {sizeof(u.rows), sizeof(u.product), sizeof(u.map), sizeof(u.gather)};
  for (int64_t i = 0; i < n; ++i) {
    const qmm_step& s = steps[i];
    if (s.kind < QMM_STEP_ROWS || s.kind > QMM_STEP_GATHER || s.bytes < 0 || (size_t)s.bytes != sizes[s.kind] || s.skip < 0 || !s.program || (s.patches && !s.patch))
      return moe_fail(QMM_ERR_BAD_ARGUMENT, "step");
    memcpy(&u, s.program, (size_t)s.bytes);
    for (int j = 0; j < s.patches; ++j) {
      const qmm_patch& q = s.patch[j];
      if (q.at < 0 || q.at > s.bytes - 8 || q.value < 0 || q.value >= n_values) return moe_fail(QMM_ERR_BAD_ARGUMENT, "step: patch");
      const uint64_t v = values[q.value] + (uint64_t)q.add;
      memcpy(reinterpret_cast<char*>(&u) + q.at, &v, 8);
    }
    int rc;
    if (s.kind == QMM_STEP_PAIR_PRODUCT) {
      rc = qmm_pair_product_run(&u.product, stream);
      if (rc == QMM_OK) i += s.skip;
      if (rc == QMM_ERR_UNSUPPORTED) rc = QMM_OK;
    } else if (s.kind == QMM_STEP_ROWS) {
      rc = qmm_row_program_run(&u.rows, stream);
    } else if (s.kind == QMM_STEP_MAP) {
      rc = qmm_pair_map_run(&u.map, stream);
    } else {
      const qmm_pair_gather& g = u.gather;
      rc = qmm_gather_qmm(g.x, g.x_dtype, g.w, g.scales, g.biases, (int)g.table_dtype, g.y, g.y_dtype, g.lhs_idx, g.rhs_idx, g.pairs,
                          g.rows, g.experts, g.n, g.k, (int)g.group_size, (int)g.bits, (int)g.mode, g.workspace,
                          (size_t)g.workspace_bytes, stream);
    }
    if (rc) return rc;
  }
  return QMM_OK;
}

}  // extern "C"
