// C ABI of libqmm_hip.so: argument validation and regime dispatch.
// See include/qmm_hip.h for the contract of every entry point.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <mutex>

#include "qmm_common.hpp"

namespace qmm {

void gemv_dispatch(const void* x, const void* w, const void* s, const void* b, int tab, void* y,
                   int y_dtype, int64_t batch, int64_t M, int64_t N, int64_t K, int gs, int bits,
                   int mode, const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t n_experts,
                   int64_t n_xrows, hipStream_t st);
void gemv_geometry(int64_t M, int64_t N, int64_t K, int* t, int* waves);
void mxfp4_geometry(int terms, int64_t batch, int64_t M, int64_t N, int64_t K, const void* s, int64_t products, int* t, int* waves);
void skinny_geometry(int64_t N, int64_t K, int bits, int* waves, int* rows_per_wg);
bool skinny2_plan(int64_t M, int64_t N, int64_t K, int bits, int* rows_per_wg);
bool skinny2_ragged_supported(int64_t N, int64_t K, int gs, int bits, int tab, const void* s, const void* b,
                              int64_t products);
int64_t skinny2_ragged_rows(int64_t N, int64_t K, int64_t products);
int64_t skinny2_g32_rows(int64_t N, int64_t K, int64_t products);
bool skinny2_g32_supported(int64_t N, int64_t K, int gs, int bits, int tab, const void* s, const void* b, int64_t products);
int device_cus();
bool skinny2_mx_plan(int64_t N, int64_t K, int* rows_per_wg);
bool skinny2_grouped_supported(int64_t N, int64_t K, int gs, int bits, int mode, int tab,
                               const void* s, const void* b, int64_t E, int64_t least_slices);
void skinny2_grouped_dispatch(const void* x, const void* w, const void* s, const void* b, void* y,
                              int y_dtype, const int32_t* segments, const int32_t* src_row,
                              const int32_t* out_row, int64_t P, int64_t T, int64_t E, int64_t N,
                              int64_t K, int gs, int bits, int mode, int tab, const int32_t* lhs_idx,
                              const int32_t* rhs_idx, hipStream_t st);
int64_t skinny2_max_segments(int64_t P, int64_t E);
void gemm_dispatch(const void* x, const void* w, const void* s, const void* b, int tab, void* y,
                   int y_dtype, const int32_t* row_offsets, const int32_t* lhs_idx,
                   const int32_t* out_idx, int64_t R, int64_t x_rows, int64_t E, int64_t N,
                   int64_t K, int gs, int bits, int mode, hipStream_t st);
int64_t gemm_row_tile(int64_t R, int64_t E);
bool gemv_runs_general(int64_t N, int64_t K, int gs, int bits, int mode, int tab, const void* s, const void* b,
                       int64_t products);
void gemv_terms_dispatch(const void* x, int x_dtype, const void* w, const void* s, void* y, int y_dtype, int64_t batch,
                         int64_t M, int64_t N, int64_t K, const int32_t* lhs_idx, const int32_t* rhs_idx,
                         const int32_t* segments, const int32_t* src_row, const int32_t* out_row, int64_t n_experts,
                         int64_t x_rows, int pairs_here, hipStream_t st);
void gemv_grouped_dispatch(const void* x, const void* w, const void* s, const void* b, int tab, void* y,
                           int y_dtype, const int32_t* segments, const int32_t* src_row,
                           const int32_t* out_row, const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t pairs,
                           int64_t n_experts, int64_t max_segments, int64_t x_rows, int64_t N,
                           int64_t K, int gs, int bits, int mode, hipStream_t st);
bool gemm2_supported(int64_t R, int64_t N, int64_t K);
size_t gemm2_workspace_bytes(int64_t R, int64_t K);
void gemm2_dispatch(const void* x, const void* w, const void* s, const void* b, int tab, void* y,
                    int y_dtype, const int32_t* row_offsets, const int32_t* lhs_idx,
                    const int32_t* out_idx, int64_t R, int64_t x_rows, int64_t E, int64_t N,
                    int64_t K, int gs, int bits, int mode, int row_tile, void* workspace,
                    size_t workspace_bytes, const ClearArgs& clear, hipStream_t st);
double gemm2s_plan(int64_t R, int64_t E, int64_t N, int64_t K, size_t part_bytes, int* tile_rows, int* splits);
double gemm2_us(int64_t R, int64_t E, int64_t N, int64_t K, size_t part_bytes);
size_t gemm2_split_workspace_bytes(int64_t R, int64_t N, int64_t K);
int short_terms(int x_dtype, int tab, int gs, int mode);
bool short_supported(int64_t R, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab, int terms,
                     const void* s, const void* b);
double short_us(int64_t R, int64_t E, int64_t N, int64_t K, int bits, int mode, int terms, size_t part_bytes);
void short_geometry(int64_t R, int64_t N, int64_t K, int bits, int mode, int* grid);
size_t short_prep_bytes(int64_t R, int64_t K, int terms);
size_t short_workspace_bytes(int64_t R, int64_t N, int64_t K, int bits, int mode, int terms);
void short_dispatch(const void* x, int x_dtype, const void* w, const void* s, const void* b, int tab, void* y,
                    int y_dtype, const int32_t* row_offsets, const int32_t* lhs_idx, const int32_t* out_idx, int64_t R,
                    int64_t x_rows, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, void* workspace,
                    size_t workspace_bytes, hipStream_t st);
bool mxfp4_mfma_supported(int64_t R, int64_t N, int64_t K);
size_t mxfp4_workspace_bytes(int64_t R, int64_t K);
double mxfp4_us(int64_t R, int64_t E, int64_t N, int64_t K);
void mxfp4_geometry(int64_t R, int64_t N, int64_t K, int* grid, int* block);
void mxfp4_mfma_dispatch(const void* x, const void* w, const void* s, void* y, int y_dtype,
                         const int32_t* row_offsets, const int32_t* lhs_idx,
                         const int32_t* out_idx, int64_t R, int64_t x_rows, int64_t E, int64_t N,
                         int64_t K, void* workspace, hipStream_t st);
void unpack_dispatch(const void* w, void* codes, int64_t rows, int64_t K, int bits, hipStream_t st);
void pack_dispatch(const void* codes, void* w, int64_t rows, int64_t K, int bits, hipStream_t st);
void dequant_dispatch(const void* w, const void* s, const void* b, int tab, void* out,
                      int out_dtype, int64_t rows, int64_t K, int gs, int bits, int mode,
                      hipStream_t st);
void take_dispatch(const void* x, int x_dtype, const int32_t* perm, void* out, int64_t rows,
                   int64_t K, hipStream_t st);
void split_terms_dispatch(const void* x, int x_dtype, void* out, int64_t batch, int64_t rows,
                          int64_t K, const int32_t* src_row, int64_t x_rows, hipStream_t st);
void sum_terms_dispatch(const void* part, int terms, void* y, int y_dtype, int64_t batch,
                        int64_t rows, int64_t N, const int32_t* offsets,
                        const int32_t* expert_of_row, int64_t E, hipStream_t st);

namespace {

thread_local char g_err[512] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int check_launch(const char* what) {
  hipError_t e = setup_error();                   // a failed launch set-up (nothing was launched)
  setup_error() = hipSuccess;
  if (e == hipSuccess) e = hipGetLastError();
  if (e != hipSuccess) return fail(QMM_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
  return QMM_OK;
}

}  // namespace

int moe_fail(int code, const char* what) { return fail(code, "%s", what); }
int moe_launched(const char* what) { return check_launch(what); }

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// Largest M served by the decode kernel.
constexpr int64_t kGemvMaxM = 16;
// Pairs at or below which the gather form runs one decode launch per pair
// instead of sorting rows by expert.
constexpr int64_t kGatherGemvMaxPairs = 64;
// From this many pairs on (and up to kGatherGemvMaxPairs) the pairs are sorted
// by expert and every expert's weight is streamed once (grouped decode); below
// it the sort's launch costs more than a shared expert saves.
constexpr int64_t kGroupedDecodeMinPairs = 4;

// Are these few pairs for the grouped decode whose workgroups sort them by
// themselves (where it serves the shape)?  Otherwise every pair is a decode
// product of its own.  From four pairs on; four-bit affine weights of
// whole slices from two, unless the result is narrow (2 pairs over 16 of 2048 x
// 4032: 6.7 / 7.1); with less than eight whole K-slices the per-pair products
// are short and it takes more pairs (us, per pair or after a sort's launch /
// here: four-bit, 8 experts of 4096 x 4096, 2 pairs 10.9 / 8.3, 16 pairs 36.9 /
// 16.7; 16 of 1024 x 8192, 3 pairs 7.9 / 9.0, 4 pairs 15.4 / 9.3; 32 of 1024 x
// 2048, 4 pairs 5.6 / 6.1, 6 pairs 8.8 / 7.0; MXFP4, 32 of 5760 x 2880, 3 pairs
// 11.2 / 11.9, 4 pairs 22.5 / 13.3; 32 of 1024 x 2048, 32 pairs 10.4 / 11.4, 64
// pairs 19.0 / 14.5).
bool sorted_here_pairs(int64_t P, int64_t N, int64_t K, int bits, int mode) {
  if (P > kGatherGemvMaxPairs) return false;
  const bool mx = mode == QMM_MODE_MXFP4;
  const int64_t row = K * (mx ? 4 : bits) / 8;
  if (row % 256 == 0 && row < 8 * 256) return P >= (mx ? 48 : 6);
  return P >= (!mx && bits == 4 && N >= 2048 && row % 256 == 0 ? 2 : 4);
}

int check_quant(int64_t N, int64_t K, int gs, int bits, int mode, int tab, const void* w,
                const void* s, const void* b) {
  if (!w || !s) return fail(QMM_ERR_BAD_ARGUMENT, "null weight or scale pointer");
  if (N < 0 || K < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (mode == QMM_MODE_MXFP4) {
    if (bits != 4) return fail(QMM_ERR_UNSUPPORTED, "mxfp4 requires bits=4, got %d", bits);
    if (gs != 32) return fail(QMM_ERR_UNSUPPORTED, "mxfp4 requires group_size=32, got %d", gs);
    if (b) return fail(QMM_ERR_BAD_ARGUMENT, "mxfp4 takes no biases");
  } else if (mode == QMM_MODE_AFFINE) {
    if (bits != 4 && bits != 8) return fail(QMM_ERR_UNSUPPORTED, "affine bits=%d (4 or 8 built)", bits);
    if (gs != 32 && gs != 64 && gs != 128)
      return fail(QMM_ERR_UNSUPPORTED, "group_size=%d (32, 64 or 128)", gs);
    if (!b) return fail(QMM_ERR_BAD_ARGUMENT, "affine mode needs biases");
    if (tab != QMM_F32 && tab != QMM_BF16 && tab != QMM_F16)
      return fail(QMM_ERR_UNSUPPORTED, "table dtype %d", tab);
  } else {
    return fail(QMM_ERR_UNSUPPORTED, "mode %d", mode);
  }
  if (K % 32) return fail(QMM_ERR_BAD_SHAPE, "K=%lld is not a multiple of 32", (long long)K);
  if (K % gs) return fail(QMM_ERR_BAD_SHAPE, "K=%lld is not a multiple of group_size=%d", (long long)K, gs);
  if (!aligned16(w)) return fail(QMM_ERR_BAD_ARGUMENT, "weight pointer not 16-byte aligned");
  return QMM_OK;
}

int check_io(const void* x, int x_dtype, void* y, int y_dtype) {
  if (!x || !y) return fail(QMM_ERR_BAD_ARGUMENT, "null activation or output pointer");
  if (x_dtype != QMM_BF16 && x_dtype != QMM_F16 && x_dtype != QMM_F32)
    return fail(QMM_ERR_UNSUPPORTED, "activation dtype %d", x_dtype);
  if (y_dtype != QMM_BF16 && y_dtype != QMM_F32 && y_dtype != QMM_F16)
    return fail(QMM_ERR_UNSUPPORTED, "output dtype %d", y_dtype);
  if (!aligned16(x)) return fail(QMM_ERR_BAD_ARGUMENT, "activation pointer not 16-byte aligned");
  return QMM_OK;
}

// ---- routing for the gather form: pairs -> rows sorted by expert -----------
// workspace layout (int32): row_offsets[E+1] | cursor[E] | src_row[P] | out_row[P] | segments
// segments (grouped decode only): [0] = count, then (expert, first sorted
// position, rows <= 16) per chunk of sixteen rows of every expert that has rows
__global__ __launch_bounds__(1024) void route_kernel(const int32_t* __restrict__ lhs_idx,
                                                     const int32_t* __restrict__ rhs_idx, int P,
                                                     int E, int32_t* __restrict__ row_offsets,
                                                     int32_t* __restrict__ cursor,
                                                     int32_t* __restrict__ src_row,
                                                     int32_t* __restrict__ out_row,
                                                     int32_t* __restrict__ segments) {
  for (int e = threadIdx.x; e <= E; e += blockDim.x) {
    row_offsets[e] = 0;
    if (e < E) cursor[e] = 0;
  }
  // slots that no valid pair lands in (pairs naming an expert outside [0, E)) gather nothing
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    src_row[p] = -1;
    out_row[p] = -1;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    const int e = rhs_idx[p];
    if (e >= 0 && e < E) atomicAdd(&cursor[e], 1);
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int run = 0;
    for (int e = 0; e < E; ++e) {
      const int c = cursor[e];
      row_offsets[e] = run;
      cursor[e] = run;
      run += c;
    }
    row_offsets[E] = run;
    if (segments) {
      int n = 0;
      for (int e = 0; e < E; ++e) {
        const int lo = row_offsets[e], cnt = row_offsets[e + 1] - lo;
        for (int c = 0; c * 16 < cnt; ++c) {
          segments[1 + 3 * n] = e;
          segments[2 + 3 * n] = lo + 16 * c;
          segments[3 + 3 * n] = cnt - 16 * c < 16 ? cnt - 16 * c : 16;
          ++n;
        }
      }
      segments[0] = n;
    }
  }
  __syncthreads();
  for (int p = threadIdx.x; p < P; p += blockDim.x) {
    const int e = rhs_idx[p];
    if (e < 0 || e >= E) continue;
    const int pos = atomicAdd(&cursor[e], 1);
    // (the indices are read twice, to count and to place: were the caller to change them meanwhile, a
    // slot past the expert's counted range would run into the next array -- such a pair is dropped)
    if (pos >= row_offsets[e + 1]) continue;
    src_row[pos] = lhs_idx ? lhs_idx[p] : p;
    out_row[pos] = p;
  }
}

// The same for up to kRoutePairs pairs and kRouteExperts experts, counted and placed
// in LDS: every thread keeps its pairs' experts, an expert's counter hands out the
// ranks, and one wavefront sums the counters, 64 experts a turn.  (The form above
// walks the experts one after the other in global memory, a round trip each.  Whole
// products, us: 256 pairs over 32 experts of 1024 x 2048 25.4 -> 20.4, 1024 pairs over
// 8 of 4096 x 4096 72.1 -> 60.3.)
constexpr int kRoutePairs = 4096, kRouteExperts = 1024, kRouteKept = kRoutePairs / 1024;

__global__ __launch_bounds__(1024) void route_lds_kernel(const int32_t* __restrict__ lhs_idx,
                                                         const int32_t* __restrict__ rhs_idx, int P,
                                                         int E, int32_t* __restrict__ row_offsets,
                                                         int32_t* __restrict__ src_row,
                                                         int32_t* __restrict__ out_row,
                                                         int32_t* __restrict__ segments) {
  __shared__ int32_t count[kRouteExperts], first[kRouteExperts];
  __shared__ int32_t total;
  const int tid = threadIdx.x;
  int ex[kRouteKept], src[kRouteKept], rank[kRouteKept];
#pragma unroll
  for (int i = 0; i < kRouteKept; ++i) {
    const int p = tid + 1024 * i;
    ex[i] = p < P ? rhs_idx[p] : -1;
    if (ex[i] >= E) ex[i] = -1;
    src[i] = p < P && lhs_idx ? lhs_idx[p] : p;
  }
  count[tid] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kRouteKept; ++i) rank[i] = ex[i] >= 0 ? atomicAdd(&count[ex[i]], 1) : 0;
  __syncthreads();
  if (tid < 64) {
    int run = 0, segs = 0;                        // rows, segments before the 64 experts of this turn
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int e = e0 + tid, c = e < E ? count[e] : 0, sg = (c + 15) / 16;
      int rows = c, upto = sg;                    // sums over the lanes up to this one
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int r = __shfl_up(rows, d), u = __shfl_up(upto, d);
        if (tid >= d) { rows += r; upto += u; }
      }
      const int lo = run + rows - c;
      if (e < E) {
        first[e] = lo;
        row_offsets[e] = lo;
        if (segments)
          for (int k = 0, n = segs + upto - sg; k < sg; ++k, ++n) {
            segments[1 + 3 * n] = e;
            segments[2 + 3 * n] = lo + 16 * k;
            segments[3 + 3 * n] = c - 16 * k < 16 ? c - 16 * k : 16;
          }
      }
      run += __shfl(rows, 63);
      segs += __shfl(upto, 63);
    }
    if (tid == 0) {
      row_offsets[E] = run;
      if (segments) segments[0] = segs;
      total = run;
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kRouteKept; ++i) {
    const int p = tid + 1024 * i;
    if (ex[i] >= 0) {
      const int pos = first[ex[i]] + rank[i];
      src_row[pos] = src[i];
      out_row[pos] = p;
    }
    // slots that no valid pair lands in (pairs naming an expert outside [0, E)) gather nothing
    if (p >= total && p < P) src_row[p] = out_row[p] = -1;
  }
}

void route(const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t E, int32_t* row_offsets,
           int32_t* cursor, int32_t* src_row, int32_t* out_row, int32_t* segments, hipStream_t st) {
  if (P <= kRoutePairs && E <= kRouteExperts)
    hipLaunchKernelGGL(route_lds_kernel, dim3(1), dim3(1024), 0, st, lhs_idx, rhs_idx, (int)P, (int)E, row_offsets,
                       src_row, out_row, segments);
  else
    hipLaunchKernelGGL(route_kernel, dim3(1), dim3(1024), 0, st, lhs_idx, rhs_idx, (int)P, (int)E, row_offsets, cursor,
                       src_row, out_row, segments);
}

size_t route_bytes(int64_t P, int64_t E) {     // a multiple of 256: what follows stays aligned
  return ((size_t)(2 * E + 1 + 2 * P) * sizeof(int32_t) + 255) / 256 * 256;
}

// the sort's arrays plus the segment list of the grouped decode
size_t route_bytes_segments(int64_t P, int64_t E) {
  return ((size_t)(2 * E + 1 + 2 * P + 1 + 3 * skinny2_max_segments(P, E)) * sizeof(int32_t) + 255) / 256 * 256;
}

// Pairs up to which the grouped decode (one decode product per expert and
// sixteen pairs) is taken: 8 experts of 14336 x 4096, 128 pairs 94 us here, 256
// pairs 120 us and 512 pairs 163 us on the row-group kernels; 32 experts of 2048 x
// 4096, 256 pairs 44 us and 512 pairs 63 us here.
bool grouped_decode_pairs(int64_t P, int64_t E) {
  static const int64_t gd_max = experiment_env("QMM_GD_MAX") ? atoll(experiment_env("QMM_GD_MAX")) : 0;
  if (P < kGroupedDecodeMinPairs) return false;
  return gd_max ? P <= gd_max : P <= 16 * E && P <= 4096;
}

// Are these pairs for the grouped decode behind a sort's launch?  (`workspace_bytes`
// hold the sort's arrays and the segment list.)
bool grouped_decode_serves(int64_t P, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab,
                           const void* s, const void* b, size_t workspace_bytes) {
  static const bool off = experiment_env("QMM_NO_GROUPED_DECODE") != nullptr;
  // Groups of 32 decode more slowly: past 64 pairs, with more than ten an expert, the
  // row-group kernels are ahead (us, here / there: 100 pairs over 8 experts of 4096 x 4096
  // 38.5 / 34.2, 500 over 32 of 1024 x 4096 43.9 / 34.9, 256 over 16 of 4096 x 2048 46.5 / 40.7;
  // 300 over 32 of 2048 x 2048 33.3 / 37.4, 128 over 32 32.4 / 35.9).
  if (mode == QMM_MODE_AFFINE && gs == 32 && P > kGatherGemvMaxPairs && P > 10 * E) return false;
  // Fewer than sixteen stay decode products of their own until what these would stream is
  // worth the sort's launch (us, here / there: 13 pairs over 4 experts of 296 x 3072, 6 MB, 8.8 /
  // 7.8, 15 of 472 x 5376, 19 MB, 11.7 / 12.5, 13 of 1312 x 2624, 22 MB, 10.8 / 13.0, 12 over 16 of 2792 x
  // 1152, 19 MB, 16.6 / 24.3).
  if (mode == QMM_MODE_AFFINE && gs == 32 && P < 16 && P * (N * K * bits / 8) <= (16 << 20)) return false;
  return grouped_decode_pairs(P, E) && !off && workspace_bytes >= route_bytes_segments(P, E) &&
         skinny2_grouped_supported(N, K, gs, bits, mode, tab, s, b, E, 8);
}

// Are these pairs for the grouped decode whose workgroups sort them by themselves?
bool sorted_here_serves(int64_t P, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab,
                        const void* s, const void* b) {
  // (float32 tables of groups of 64, and groups of 32, leave no LDS for the sort)
  return sorted_here_pairs(P, N, K, bits, mode) && E > 0 && !(mode == QMM_MODE_AFFINE && ((tab == QMM_F32 && gs == 64) || gs == 32)) &&
         skinny2_grouped_supported(N, K, gs, bits, mode, tab, s, b, E, 3);
}

// From sixteen pairs on, and half a pair an expert, shapes that only the
// general decode kernels serve are grouped by expert as well: an expert's
// weights are then read once for up to sixteen of its pairs instead of
// once per pair.  (The sort costs a launch of its own, and with fewer
// pairs than that few of them share an expert.  Measured on 32 MXFP4
// experts of [5760, 2880]: 16 pairs 61 against 60 us, 32 pairs 86 against
// 110, 64 pairs 109 against 216; on 128 experts: 32 pairs 128 against 110,
// 64 pairs 194 against 217; 8 experts of [4096, 11008] with four-bit
// codes: 16 pairs 108 against 206 us, 32 pairs 110 against 397.)
bool sorts_general(int64_t P, int64_t E, size_t workspace_bytes) {
  return P >= 16 && 2 * P >= E && grouped_decode_pairs(P, E) && workspace_bytes >= route_bytes_segments(P, E);
}

// More pairs whose K is no multiple of 64 (groups of 32): neither the re-laying kernels
// nor the short-group one takes them, and the row-group kernel that does walks K in a
// workgroup a tile.  The general decode kernels behind a sort's launch read an expert's
// weight once for sixteen of its pairs (us, here / on row groups; 8 experts of 4096 x 992,
// four-bit affine codes: 65 pairs 22 / 53, 256 46 / 61, 512 80 / 69, 16 of 1024 x 480:
// 512 pairs 23.9 / 23.4; MXFP4: 65 17 / 76, 512 60 / 93, 1024 109 / 129, float32 rows in one
// launch instead of one a term and more 23 / 233, 102 / 299, 189 / 423).
constexpr int64_t kOddPairs = 2048;

bool sorts_odd(int64_t P, int64_t E, int64_t N, int64_t K, int mode, size_t workspace_bytes) {
  return P > kGatherGemvMaxPairs && P <= kOddPairs && P <= (mode == QMM_MODE_MXFP4 ? 64 : 24) * E && K % 64 != 0 && E <= 65535 &&
         N <= INT32_MAX && K <= INT32_MAX && workspace_bytes >= route_bytes_segments(P, E);
}

// The general kernels sort up to 64 pairs themselves: a few instructions an expert that
// occurs, in every workgroup, against a launch ahead of the product.  By how many there
// are of both (us, here / behind the launch: 64 pairs over 8 experts of 1024 x 1024, 9200,
// 8.4 / 11.5, over 8 of 6528 x 1024, 58750, 27.3 / 29.2, 16 over 32 of 2048 x 992, 37000, 12.0 / 13.8,
// 24 of it, 80000, 15.8 / 15.8, 32 of it, 148000, 21.6 / 19.1; MXFP4, bf16 activations).
bool sorts_itself(int64_t P, int64_t E, int64_t N) {
  const int64_t segments = skinny2_max_segments(P, E);
  return P <= kGatherGemvMaxPairs && segments * segments * ((N + 15) / 16) <= (1 << 16);
}

bool grouped_general_serves(int64_t P, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab,
                            const void* s, const void* b, size_t workspace_bytes) {
  return sorts_general(P, E, workspace_bytes) && gemv_runs_general(N, K, gs, bits, mode, tab, s, b, E) && !experiment_env("QMM_NO_GROUPED_GEMV");
}

// ---- float16 / float32 activations ---------------------------------------------
// The kernels multiply bf16 operands.  Wider activations are split, exactly,
// into bf16 terms (float16: two, float32: three), every term is multiplied
// like a bf16 activation (products exact, float32 accumulate) and the terms'
// float32 results are added, largest first, before the one rounding to the
// output type.  In the dense decode case the terms ride as extra rows of the
// same launch (terms x M <= 16: the weight is still streamed once).
int act_terms(int x_dtype) { return x_dtype == QMM_F32 ? 3 : x_dtype == QMM_F16 ? 2 : 1; }

// The general MXFP4 decode kernel splits the rows itself, one launch where the
// loader-wavefront kernel needs the split and the sum round it (three, and one or two a
// term for pairs that it sorts); but it reads the weight more slowly.  By the bytes that
// it would stream, then (us, float32, here / there):
//   rows, pairs of their own: 4096 x 4096 9.3 / 13.2, two pairs of it 14.2 / 14.0, 8 of
//   1024 x 2048 9.7 / 14.0, 32 of 16 experts of it (19 MB) 17.7 / 15.5, 4096 x 11008 21.3 / 13.9;
//   64 pairs of 16 experts of 1024 x 2048 (21 MB, a third of what pairs of their own
//   stream) 19.2 / 32.7;
//   sorted pairs: 8 of 32 experts of 2880 x 2880 (33 MB) 26.4 / 35.6, 64 of 8 of 2880 x
//   1088 22.0 / 36.8, 8 of 8 of 4096 x 4096 (67 MB) 45.4 / 39.0;
//   past 64 pairs, against the row-group kernels: 78 of 8 of 1024 x 1024 (6.3 MB) 11.7 /
//   15.4 (float16 11.0 / 14.3), 128 of it (8.4) 15.5 / 15.7 (11.4 / 16.3) (a K that is no
//   multiple of 64: sorts_odd) -- into 16-bit results: those kernels' sums over parts of K
//   are the more exact ones (float32 results, 96 pairs of 280 x 1024 6.9e-8 / 6.1e-8 from
//   64 bits, 134 of 352 x 1408 7.8e-8 / 6.6e-8).
constexpr int64_t kTermsBytes = 12 << 20, kTermsBytesMost = 34 << 20, kTermsBytesManyPairs = 18 << 20;

// A wavefront adds up its share of K in one accumulator a term.  Eight of them to about 5120
// codes are as exact as the loader-wavefront kernel, beyond it their sums come out less
// exact and later (float32 rows, distance from 64 bits, here / there: 0.98e-7 / 0.98e-7 up to K =
// 4096, within 8 % either way by the rows up to 5120, 1.16e-7 / 1.04e-7 at 6464, 1.25e-7 / 1.04e-7
// at 8192, 1.55e-7 / 1.06e-7 at 13312).  Against its own launches round the general kernel,
// whose sums are the same, it holds to 6144 (us: 1744 x 6048 13.4 / 14.1, 1416 x 7136 14.9 / 13.7,
// 784 x 11424 20.5 / 15.8, float16 4040 x 6112 10.7 / 12.8, 2216 x 8672 15.2 / 14.3).
constexpr int64_t kTermsCodes = 5120, kTermsCodesGeneral = 6144;

// Dense rows split in the kernel, where the loader-wavefront kernel serves the shape too
// (us a call, here / there): with two workgroups a compute unit, half the wavefronts each, by
// the bytes (12688 x 1472 float16 10.4 / 11.8, float32 8232 x 1216 9.7 / 11.6, 13800 x 1216 10.4 /
// 11.8, 12992 x 1920 12.8 / 10.9, but 0.73e-7 from 64 bits against 0.85e-7), past 2048 codes while
// the workgroups are one round (float32 3904 x 4032 9.2 / 12.3, 2296 x 3648 9.7 / 12.9; 4408 x
// 4032 15.1 / 13.1, 9416 x 2432 18.4 / 11.9).
bool terms_dense(int64_t batch, int64_t N, int64_t K) {
  if (K <= 2048) return N * K / 2 <= kTermsBytes / batch;
  return K <= kTermsCodes && batch * ceil_div(N, 16) <= device_cus();
}

bool terms_in_kernel(const void* x, int terms, int64_t P, int64_t E, int64_t N, int64_t K, int gs, int bits, int mode, int tab,
                     const void* s, const void* b, int y_dtype, size_t workspace_bytes) {
  if (mode != QMM_MODE_MXFP4 || !aligned16(x) || P <= 0 || E > 65535 || N > INT32_MAX || K > INT32_MAX || N * K >= (1ll << 40))
    return false;
  const bool sorted = sorts_general(P, E, workspace_bytes);
  if (P > kGatherGemvMaxPairs && !sorted) return false;
  const int64_t bytes = (sorted ? skinny2_max_segments(P, E) : P) * (N * K / 2);
  if (P > kGatherGemvMaxPairs) return y_dtype != QMM_F32 && terms * bytes <= (K < 512 ? kTermsBytes : kTermsBytesManyPairs);
  if (gemv_runs_general(N, K, gs, bits, mode, tab, s, b, E)) return sorted || K <= kTermsCodesGeneral;
  if (K > kTermsCodes) return false;
  if (sorted_here_serves(P, E, N, K, gs, bits, mode, tab, s, b) ||
      grouped_decode_serves(P, E, N, K, gs, bits, mode, tab, s, b, workspace_bytes))
    return bytes <= kTermsBytesMost;
  return bytes <= kTermsBytes || (bytes <= kTermsBytesMost && P * (N * K / 2) >= 3 * bytes);
}

}  // namespace

// How the general MXFP4 decode kernel would take these pairs: 1 each a product of its
// own, 2 sorted by the kernel itself, 0 not at all (another kernel, or the sort's launch).
// `waves`: how many wavefronts share the contraction there.
int pair_product_route(const void* x, int x_dtype, int64_t P, int64_t E, int64_t N, int64_t K, const void* s, int y_dtype, int* waves) {
  if (P <= 0 || P > kGatherGemvMaxPairs || !aligned16(x)) return 0;
  const int terms = act_terms(x_dtype);
  const size_t any = ~(size_t)0 / 4;               // (the route of a call with all the scratch it asks for)
  if (terms > 1 ? !terms_in_kernel(x, terms, P, E, N, K, 32, 4, QMM_MODE_MXFP4, QMM_BF16, s, nullptr, y_dtype, any)
                : E > 65535 || N > INT32_MAX || K > INT32_MAX || N * K >= (1ll << 40) ||
                      !gemv_runs_general(N, K, 32, 4, QMM_MODE_MXFP4, QMM_BF16, s, nullptr, E))
    return 0;
  const bool sorted = sorts_general(P, E, any);
  if (sorted && !sorts_itself(P, E, N)) return 0;
  int t;
  mxfp4_geometry(terms, sorted ? skinny2_max_segments(P, E) : P, sorted ? 16 : terms, N, K, s, E, &t, waves);
  return sorted ? 2 : 1;
}

namespace {

size_t align256(size_t n) { return (n + 255) / 256 * 256; }

// Scratch of the bf16 dense / grouped product over `rows` rows.  `exact`: the
// activation terms must stay exact, so MXFP4 weights take the bf16 kernels
// (their FP6 activation terms would round).
size_t dense_scratch(int64_t rows, int64_t N, int64_t K, int mode, bool exact) {
  if (mode == QMM_MODE_MXFP4 && !exact && rows > kGemvMaxM && mxfp4_mfma_supported(rows, N, K))
    return mxfp4_workspace_bytes(rows, K);
  if (rows > kGemvMaxM && gemm2_supported(rows, N, K)) return gemm2_workspace_bytes(rows, K);
  return 0;
}

// ... with room for the sums of a split K, which the dense prefill product takes where it is there
size_t dense_scratch_split(int64_t rows, int64_t N, int64_t K, int mode, bool exact) {
  const size_t least = dense_scratch(rows, N, K, mode, exact);
  const bool mx = mode == QMM_MODE_MXFP4 && !exact && mxfp4_mfma_supported(rows, N, K);
  if (rows <= kGemvMaxM || N <= 0 || mx || !gemm2_supported(rows, N, K)) return least;
  return std::max(least, gemm2_split_workspace_bytes(rows, N, K));
}

// Float16 / float32 activations: their terms as bf16 rows and the terms' float32 products.
size_t term_bytes(int64_t terms, int64_t rows, int64_t N, int64_t K) {
  return align256((size_t)(terms * rows * K) * 2) + align256((size_t)(terms * rows * N) * 4);
}

// Is the short-group kernel the one to take?  `E` experts share the R rows
// (`grouped`; else a dense product and E = 1), the activations are `terms` bf16
// terms (`own` of the short-group kernel), and each kernel has what `scratch` leaves it for a split K's sums.  All
// kernels' times have been fitted over the shapes they serve; where they come close
// the choice matters little.  (4096 x 4096, four-bit codes: 17 rows 12 against 17 us of the
// prefill kernel, 128 rows 19 against 22, 512 rows 32 against 36; 14336 x 4096:
// 20 against 29, 31 against 34, 114 against 61.  Of 208 affine products, 48 of them
// groups, the slower kernel is taken in a few, 11 % slower at worst; of 92
// MXFP4 ones the slower is taken by 17 % at worst and by 0.6 % on average:
// profiles/prefill_plan_fits.txt.)
bool short_wins(int64_t R, int64_t E, int64_t N, int64_t K, int bits, int mode, int terms, int own, bool grouped, size_t scratch) {
  if (K % 64 || N <= 0) return false;
  if (const char* env = experiment_env("QMM_SHORT")) return env[0] != '0';
  double other, ours = 0.0;
  if (mode == QMM_MODE_MXFP4 && terms == 1 && mxfp4_mfma_supported(R, N, K)) {
    if (N < 512) return false;                   // (a few column tiles: not measured, left as it is)
    other = mxfp4_us(R, E, N, K);
  } else {
    // (row groups keep their whole K there, one product a term; dense, the terms are rows of one product)
    const size_t held = gemm2_workspace_bytes(terms * R, K) + (terms > 1 ? term_bytes(terms, R, N, K) : 0);
    other = grouped ? terms * gemm2_us(R, E, N, K, 0) : gemm2_us(terms * R, 1, N, K, scratch > held ? scratch - held : 0);
    if (terms > 1) other += 5.2 + (double)terms * R * N * 1.4e-6;
    // (the terms' own launches: float32 rows of 2387 x 11264 83 us ahead of the re-laying, 40 here;
    // for groups both times are too short by more than that)
    if (terms > 1 && !grouped) other += (double)R * K * (terms == 3 ? 3.0e-6 : 2.4e-6);
    if (own > 1 && !grouped) ours = (double)R * K * (own == 3 ? 1.4e-6 : 0.9e-6);
  }
  const size_t prep = short_prep_bytes(R, K, own);
  return ours + short_us(R, E, N, K, bits, mode, own, scratch > prep ? scratch - prep : 0) < other;
}

// Scratch that lets a short-group product over R rows run as it would best.
size_t short_scratch(int64_t R, int64_t N, int64_t K, int bits, int mode, int terms) {
  if (R <= 0 || R > 4096 || N <= 0 || K <= 0 || K % 64 || terms * R <= kGemvMaxM) return 0;
  // (float16 rows are one term or two: the tables' type is not known here)
  const size_t own = terms == 2 && mode == QMM_MODE_AFFINE ? short_workspace_bytes(R, N, K, bits, mode, 1) : 0;
  return std::max(own, short_workspace_bytes(R, N, K, bits, mode, terms));
}

size_t gather_scratch(int64_t P, int64_t E, int64_t N, int64_t K, bool exact) {
  if (P < kGroupedDecodeMinPairs) return 0;
  const size_t decode = grouped_decode_pairs(P, E) ? route_bytes_segments(P, E) : 0;
  if (P <= kGatherGemvMaxPairs) return decode;    // the expert sort of the grouped decode
  // the expert sort's arrays, then (when the register-operand kernel serves
  // the shape) the re-laid copy of the gathered activation rows
  size_t relaid = gemm2_supported(P, N, K) ? gemm2_workspace_bytes(P, K) : 0;
  if (!exact && mxfp4_mfma_supported(P, N, K) && mxfp4_workspace_bytes(P, K) > relaid)
    relaid = mxfp4_workspace_bytes(P, K);          // the mode is not known here: the larger of the two
  const size_t gemm = route_bytes(P, E) + relaid;
  return gemm > decode ? gemm : decode;
}

// ---- scratch of the allocation-free entry point ------------------------------
// Part of the code object: each GPU that loads the library holds its own copy
// at its own address.  In host code the name is only a handle for
// hipGetSymbolAddress; the address it yields is what kernels are given.
__device__ __align__(256) unsigned char scratch[QMM_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's scratch address (looked up once per device).
int static_scratch(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(QMM_ERR_HIP, "hipGetDevice: %s", hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(QMM_ERR_HIP, "device ordinal %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(QMM_ERR_HIP, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return QMM_OK;
}

}  // namespace
}  // namespace qmm

using namespace qmm;

extern "C" {

int qmm_abi_version(void) { return 2; }

const char* qmm_last_error(void) { return g_err; }

size_t qmm_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K, int, int bits, int mode,
                           int x_dtype) {
  const int terms = act_terms(x_dtype);
  const size_t sh = short_scratch(M, N, K, bits, mode, terms);
  if (terms == 1) return std::max(sh, dense_scratch_split(M, N, K, mode, false));
  // terms as bf16 rows, their float32 products, then the scratch of the bf16
  // product: over terms x M stacked rows (dense) or over M rows (grouped)
  if (batch < 1) batch = 1;
  const size_t stacked = dense_scratch_split(terms * M, N, K, mode, true), plain = dense_scratch(M, N, K, mode, true);
  return std::max(sh, term_bytes(terms, batch * M, N, K) + std::max(stacked, plain));
}

// What a gathered product needs to run at all on its preferred kernels, without
// the sums of a split K (those it takes only where there is room).
static size_t gather_minimum(int64_t P, int64_t E, int64_t N, int64_t K, int x_dtype) {
  const int terms = act_terms(x_dtype);
  if (terms == 1) return gather_scratch(P, E, N, K, false);
  // the gathered rows' terms, their float32 products, the bf16 product's scratch
  return term_bytes(terms, P, N, K) + gather_scratch(P, E, N, K, true);
}

// With the sums of a split K, up to the size of the static scratch: a caller of
// qmm_gather_qmm_static can tell from this alone whether the call will be taken.
// (Of 10 000 shapes drawn over 8 to 128 experts 191 would have asked for more, and
// the fitted time of six of them is 1 to 5 % better with it.)
size_t qmm_gather_workspace_bytes(int64_t P, int64_t E, int64_t N, int64_t K, int x_dtype) {
  const size_t least = gather_minimum(P, E, N, K, x_dtype);
  if (P <= kGatherGemvMaxPairs) return least;
  const int terms = act_terms(x_dtype);
  size_t sums = route_bytes(P, E) + std::max(short_scratch(P, N, K, 4, QMM_MODE_AFFINE, terms),
                                             short_scratch(P, N, K, 8, QMM_MODE_AFFINE, terms));
  if (K % 64 != 0 && P <= kOddPairs) sums = std::max(sums, route_bytes_segments(P, E));
  return std::max(least, std::min(sums, (size_t)QMM_STATIC_SCRATCH_BYTES));
}

int qmm_plan(int64_t M, int64_t N, int64_t K, int group_size, int bits, int mode, int* kernel,
             int* grid, int* block) {
  if (M > kGemvMaxM && short_wins(M, 1, N, K, bits, mode, 1, 1, false, ~(size_t)0)) {     // (bf16 activations and tables, ample scratch assumed)
    int g;
    short_geometry(M, N, K, bits, mode, &g);
    if (kernel) *kernel = QMM_KERNEL_GEMM;
    if (grid) *grid = g;
    if (block) *block = 512;
    return QMM_OK;
  }
  if (mode == QMM_MODE_MXFP4 && M > kGemvMaxM && mxfp4_mfma_supported(M, N, K)) {
    int g, b;
    mxfp4_geometry(M, N, K, &g, &b);
    if (kernel) *kernel = QMM_KERNEL_MXFP4_MFMA;
    if (grid) *grid = g;
    if (block) *block = b;
    return QMM_OK;
  }
  if (M <= kGemvMaxM && mode == QMM_MODE_MXFP4) {
    // the loader-wavefront kernel from three K-slices a row on, its ragged one-pass form for a K that
    // is no whole number of slices
    int rows;
    if (skinny2_mx_plan(N, K, &rows)) {
      if (kernel) *kernel = QMM_KERNEL_GEMV;
      if (grid) *grid = (int)ceil_div(N, (int64_t)rows);
      if (block) *block = 64 * 12;
      return QMM_OK;
    }
  }
  if (M <= kGemvMaxM && mode == QMM_MODE_AFFINE && (group_size == 64 || group_size == 128) &&
      (bits == 4 || bits == 8) && K % (2048 / bits) == 0) {
    // the staged decode kernel (bf16 tables assumed): contiguous row ranges
    int waves, rows, rows2;
    skinny_geometry(N, K, bits, &waves, &rows);
    // eight compute + four loader wavefronts where the loader kernel serves the shape
    const bool loaders = !experiment_env("QMM_SKINNY_V1") && skinny2_plan(M, N, K, bits, &rows2);
    if (loaders) rows = rows2;
    if (kernel) *kernel = QMM_KERNEL_GEMV;
    if (grid) *grid = (int)ceil_div(N, rows);
    if (block) *block = loaders ? 64 * 12 : 64 * waves;
    return QMM_OK;
  }
  const bool ragged = M <= kGemvMaxM && mode == QMM_MODE_AFFINE && skinny2_ragged_supported(N, K, group_size, bits, QMM_BF16, nullptr, nullptr, 1);
  if (ragged || (M <= kGemvMaxM && mode == QMM_MODE_AFFINE && skinny2_g32_supported(N, K, group_size, bits, QMM_BF16, nullptr, nullptr, 1))) {
    if (kernel) *kernel = QMM_KERNEL_GEMV;
    if (grid) *grid = (int)ceil_div(N, ragged ? skinny2_ragged_rows(N, K, 1) : skinny2_g32_rows(N, K, 1));
    if (block) *block = 64 * 12;
    return QMM_OK;
  }
  if (M <= kGemvMaxM) {
    int t, waves;
    gemv_geometry(M, N, K, &t, &waves);
    if (kernel) *kernel = QMM_KERNEL_GEMV;
    if (grid) *grid = (int)ceil_div(N, 16 * t);
    if (block) *block = 64 * waves;
  } else if (gemm2_supported(M, N, K) && (mode == QMM_MODE_MXFP4 || bits == 4 || bits == 8)) {
    // the split-role kernel (bf16 tables assumed): four multiplying and four dequantizing wavefronts
    int rows, splits;
    gemm2s_plan(M, 1, N, K, ~(size_t)0, &rows, &splits);
    if (kernel) *kernel = QMM_KERNEL_GEMM;
    if (grid) *grid = (int)(ceil_div(N, 128) * ceil_div(M, rows) * splits);
    if (block) *block = 512;
  } else {
    const int64_t bm = gemm_row_tile(M, 1);
    if (kernel) *kernel = QMM_KERNEL_GEMM;
    if (grid) *grid = (int)(ceil_div(N, 128) * ceil_div(M, bm));
    if (block) *block = 256;
  }
  return QMM_OK;
}

// One product on the short-group kernel if it serves it, arguments included: true
// when it was launched (*rc: the launches' status), false when the other kernels
// are to take it (or to say what is wrong with it).  It needs less scratch and less
// alignment than they do: the callers see to it that a call is refused whichever
// kernel would have run.
static bool ran_short(const void* x, int x_dtype, const void* w, const void* scales, const void* biases,
                      int table_dtype, void* y, int y_dtype, const int32_t* row_offsets, const int32_t* lhs_idx,
                      const int32_t* out_idx, int64_t R, int64_t x_rows, int64_t E, int64_t N, int64_t K,
                      int group_size, int bits, int mode, void* workspace, size_t workspace_bytes, void* stream,
                      int* rc) {
  const int terms = short_terms(x_dtype, table_dtype, group_size, mode);
  if (R <= 0 || E <= 0 || N <= 0 || K <= 0 || act_terms(x_dtype) * R <= kGemvMaxM || R > INT32_MAX / 2 || N > INT32_MAX ||
      K > INT32_MAX || E > 65535 ||
      !short_wins(R, E, N, K, bits, mode, act_terms(x_dtype), terms, row_offsets != nullptr, workspace_bytes))
    return false;
  if (check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases) || check_io(x, x_dtype, y, y_dtype) ||
      !workspace || !aligned16(workspace) || workspace_bytes < short_prep_bytes(R, K, terms) ||
      !short_supported(R, E, N, K, mode == QMM_MODE_MXFP4 ? 32 : group_size, bits, mode, table_dtype, terms, scales, biases))
    return false;
  short_dispatch(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, row_offsets, lhs_idx, out_idx, R, x_rows, E, N,
                 K, mode == QMM_MODE_MXFP4 ? 32 : group_size, bits, mode, workspace, workspace_bytes,
                 static_cast<hipStream_t>(stream));
  *rc = check_launch("short-group product launch");
  return true;
}

// The three products on bf16 activations.  `exact`: the activations are exact
// terms of a wider type (MXFP4 weights then take the bf16 kernels).
static int dense_bf16(const void* x, int x_dtype, const void* w, const void* scales,
                      const void* biases, int table_dtype, void* y, int y_dtype, int64_t batch,
                      int64_t M, int64_t N, int64_t K, int group_size, int bits, int mode,
                      void* workspace, size_t workspace_bytes, void* stream, bool exact) {
  if (batch < 0 || M < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (batch == 0 || M == 0 || N == 0) return QMM_OK;
  if (K == 0) return fail(QMM_ERR_BAD_SHAPE, "K=0");
  int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
  if (rc) return rc;
  rc = check_io(x, x_dtype, y, y_dtype);
  if (rc) return rc;
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || batch > 65535 || M * K >= (1ll << 30))
    return fail(QMM_ERR_BAD_SHAPE, "shape exceeds kernel index range");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (M <= kGemvMaxM) {
    gemv_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, batch, M, N, K, group_size,
                  bits, mode, nullptr, nullptr, 0, 0, st);
    return check_launch("gemv launch");
  }
  const int wbits = mode == QMM_MODE_MXFP4 ? 4 : bits;
  const int64_t wpr = K * wbits / 32;
  const int64_t ng = mode == QMM_MODE_MXFP4 ? K / 32 : K / group_size;
  const int tabsz = mode == QMM_MODE_MXFP4 ? 1 : (table_dtype == QMM_F32 ? 4 : 2);
  const int ysz = y_dtype == QMM_F32 ? 4 : 2;
  if (mode == QMM_MODE_MXFP4 && !exact && mxfp4_mfma_supported(M, N, K)) {
    // block-scaled matrix cores; the activations are split into the workspace first
    const size_t need = mxfp4_workspace_bytes(M, K);
    if (!workspace || workspace_bytes < need)
      return fail(QMM_ERR_WORKSPACE, "mxfp4 needs %zu workspace bytes, got %zu", need,
                  workspace ? workspace_bytes : (size_t)0);
    if (!aligned16(workspace) || !aligned16(scales))
      return fail(QMM_ERR_BAD_ARGUMENT, "workspace / scale pointer not 16-byte aligned");
    for (int64_t z = 0; z < batch; ++z) {
      mxfp4_mfma_dispatch(static_cast<const char*>(x) + z * M * K * 2,
                          static_cast<const uint32_t*>(w) + z * N * wpr,
                          static_cast<const char*>(scales) + z * N * ng,
                          static_cast<char*>(y) + z * M * N * ysz, y_dtype, nullptr, nullptr,
                          nullptr, M, M, 1, N, K, workspace, st);
      rc = check_launch("mxfp4 launch");
      if (rc) return rc;
    }
    return QMM_OK;
  }
  if (gemm2_supported(M, N, K)) {
    const size_t need = gemm2_workspace_bytes(M, K);
    if (!workspace || workspace_bytes < need)
      return fail(QMM_ERR_WORKSPACE, "the prefill kernel needs %zu workspace bytes, got %zu", need,
                  workspace ? workspace_bytes : (size_t)0);
    if (!aligned16(workspace) || !aligned16(scales))
      return fail(QMM_ERR_BAD_ARGUMENT, "workspace / table pointer not 16-byte aligned");
    const int bm = (int)gemm_row_tile(M, 1);
    for (int64_t z = 0; z < batch; ++z) {
      gemm2_dispatch(static_cast<const char*>(x) + z * M * K * 2,
                     static_cast<const uint32_t*>(w) + z * N * wpr,
                     static_cast<const char*>(scales) + z * N * ng * tabsz,
                     biases ? static_cast<const char*>(biases) + z * N * ng * tabsz : nullptr,
                     table_dtype, static_cast<char*>(y) + z * M * N * ysz, y_dtype, nullptr, nullptr,
                     nullptr, M, M, 1, N, K, group_size, bits, mode, bm, workspace, workspace_bytes, ClearArgs{}, st);
      rc = check_launch("gemm launch");
      if (rc) return rc;
    }
    return QMM_OK;
  }
  for (int64_t z = 0; z < batch; ++z) {
    gemm_dispatch(static_cast<const char*>(x) + z * M * K * 2,
                  static_cast<const uint32_t*>(w) + z * N * wpr,
                  static_cast<const char*>(scales) + z * N * ng * tabsz,
                  biases ? static_cast<const char*>(biases) + z * N * ng * tabsz : nullptr,
                  table_dtype, static_cast<char*>(y) + z * M * N * ysz, y_dtype, nullptr, nullptr,
                  nullptr, M, M, 1, N, K, group_size, bits, mode, st);
    rc = check_launch("gemm launch");
    if (rc) return rc;
  }
  return QMM_OK;
}

static int grouped_bf16(const void* x, int x_dtype, const void* w, const void* scales,
                        const void* biases, int table_dtype, void* y, int y_dtype,
                        const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                        int group_size, int bits, int mode, void* workspace, size_t workspace_bytes,
                        void* stream, bool exact, ClearArgs* clear) {
  if (R < 0 || E < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (R == 0 || N == 0 || E == 0) return QMM_OK;
  if (!row_offsets) return fail(QMM_ERR_BAD_ARGUMENT, "null row_offsets");
  int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
  if (rc) return rc;
  rc = check_io(x, x_dtype, y, y_dtype);
  if (rc) return rc;
  if (R > INT32_MAX || N > INT32_MAX || K > INT32_MAX || E > 65535 || R * K >= (1ll << 30))
    return fail(QMM_ERR_BAD_SHAPE, "shape exceeds kernel index range");
  if (mode == QMM_MODE_MXFP4 && !exact && mxfp4_mfma_supported(R, N, K) && workspace &&
      workspace_bytes >= mxfp4_workspace_bytes(R, K) && aligned16(workspace) && aligned16(scales)) {
    // MXFP4 experts on the block-scaled matrix cores
    mxfp4_mfma_dispatch(x, w, scales, y, y_dtype, row_offsets, nullptr, nullptr, R, R, E, N, K,
                        workspace, static_cast<hipStream_t>(stream));
    return check_launch("grouped mxfp4 launch");
  }
  if (gemm2_supported(R, N, K) && workspace && workspace_bytes >= gemm2_workspace_bytes(R, K) &&
      aligned16(workspace)) {
    gemm2_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, row_offsets, nullptr, nullptr, R,
                   R, E, N, K, group_size, bits, mode, (int)gemm_row_tile(R, E), workspace, workspace_bytes,
                   *clear, static_cast<hipStream_t>(stream));
    clear->y = nullptr;                            // done beside the re-laying
    return check_launch("grouped gemm launch");
  }
  // without a workspace the grouped product runs on the LDS-staged kernel
  gemm_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, row_offsets, nullptr, nullptr, R,
                R, E, N, K, group_size, bits, mode, static_cast<hipStream_t>(stream));
  return check_launch("grouped gemm launch");
}

static int gather_bf16(const void* x, int x_dtype, const void* w, const void* scales,
                       const void* biases, int table_dtype, void* y, int y_dtype,
                       const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t T,
                       int64_t E, int64_t N, int64_t K, int group_size, int bits, int mode,
                       void* workspace, size_t workspace_bytes, void* stream, bool exact) {
  if (P < 0 || T < 0 || E < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (P == 0 || N == 0) return QMM_OK;
  if (!rhs_idx) return fail(QMM_ERR_BAD_ARGUMENT, "null rhs_idx");
  int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
  if (rc) return rc;
  rc = check_io(x, x_dtype, y, y_dtype);
  if (rc) return rc;
  if (P > INT32_MAX / 2 || N > INT32_MAX || K > INT32_MAX || E > 65535 || T * K >= (1ll << 30))
    return fail(QMM_ERR_BAD_SHAPE, "shape exceeds kernel index range");
  hipStream_t st = static_cast<hipStream_t>(stream);
  // few pairs: the grouped decode whose workgroups sort them by themselves
  if (sorted_here_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases)) {
    skinny2_grouped_dispatch(x, w, scales, biases, y, y_dtype, nullptr, nullptr, nullptr, P, T, E, N, K,
                             group_size, bits, mode, table_dtype, lhs_idx, rhs_idx, st);
    return check_launch("grouped decode launch");
  }
  if (workspace && grouped_decode_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, workspace_bytes)) {
    int32_t* ro = static_cast<int32_t*>(workspace);
    int32_t* cursor = ro + E + 1;
    int32_t* src_row = cursor + E;
    int32_t* out_row = src_row + P;
    int32_t* segments = out_row + P;
    route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, segments, st);
    rc = check_launch("route launch");
    if (rc) return rc;
    skinny2_grouped_dispatch(x, w, scales, biases, y, y_dtype, segments, src_row, out_row, P, T, E, N, K,
                             group_size, bits, mode, table_dtype, nullptr, nullptr, st);
    return check_launch("grouped decode launch");
  }
  if (P <= kGatherGemvMaxPairs) {
    if (workspace && grouped_general_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, workspace_bytes)) {
      if (sorts_itself(P, E, N)) {
        gemv_grouped_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, nullptr, nullptr, nullptr, lhs_idx, rhs_idx, P, E,
                              skinny2_max_segments(P, E), T, N, K, group_size, bits, mode, st);
        return check_launch("grouped gemv launch");
      }
      int32_t* ro = static_cast<int32_t*>(workspace);
      int32_t* cursor = ro + E + 1;
      int32_t* src_row = cursor + E;
      int32_t* out_row = src_row + P;
      int32_t* segments = out_row + P;
      route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, segments, st);
      rc = check_launch("route launch");
      if (rc) return rc;
      gemv_grouped_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, segments, src_row, out_row, nullptr, nullptr, 0, E,
                            skinny2_max_segments(P, E), T, N, K, group_size, bits, mode, st);
      return check_launch("grouped gemv launch");
    }
    gemv_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, P, 1, N, K, group_size, bits,
                  mode, lhs_idx, rhs_idx, E, T, st);
    return check_launch("gather gemv launch");
  }
  if (workspace && sorts_odd(P, E, N, K, mode, workspace_bytes)) {
    int32_t* ro = static_cast<int32_t*>(workspace);
    int32_t* cursor = ro + E + 1;
    int32_t* src_row = cursor + E;
    int32_t* out_row = src_row + P;
    int32_t* segments = out_row + P;
    route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, segments, st);
    rc = check_launch("route launch");
    if (rc) return rc;
    gemv_grouped_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, segments, src_row, out_row, nullptr, nullptr, 0, E,
                          skinny2_max_segments(P, E), T, N, K, group_size, bits, mode, st);
    return check_launch("grouped gemv launch");
  }
  const size_t need = route_bytes(P, E);
  if (!workspace || workspace_bytes < need)
    return fail(QMM_ERR_WORKSPACE, "gather_qmm needs %zu workspace bytes, got %zu", need,
                workspace_bytes);
  int32_t* ro = static_cast<int32_t*>(workspace);
  int32_t* cursor = ro + E + 1;
  int32_t* src_row = cursor + E;
  int32_t* out_row = src_row + P;
  route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, nullptr, st);
  rc = check_launch("route launch");
  if (rc) return rc;
  if (ran_short(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, ro, src_row, out_row, P, T, E, N, K, group_size,
                bits, mode, static_cast<char*>(workspace) + need, workspace_bytes - need, stream, &rc))
    return rc;
  if (mode == QMM_MODE_MXFP4 && !exact && mxfp4_mfma_supported(P, N, K) &&
      workspace_bytes >= need + mxfp4_workspace_bytes(P, K) && aligned16(workspace) &&
      aligned16(scales)) {
    mxfp4_mfma_dispatch(x, w, scales, y, y_dtype, ro, src_row, out_row, P, T, E, N, K,
                        static_cast<char*>(workspace) + need, st);
    return check_launch("gather mxfp4 launch");
  }
  if (gemm2_supported(P, N, K) && workspace_bytes >= need + gemm2_workspace_bytes(P, K) &&
      aligned16(workspace)) {
    // rows gathered in expert order into the re-laid copy, results scattered back to pair order
    gemm2_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, ro, src_row, out_row, P, T, E, N, K,
                   group_size, bits, mode, (int)gemm_row_tile(P, E),
                   static_cast<char*>(workspace) + need, workspace_bytes - need, ClearArgs{}, st);
    return check_launch("gather gemm launch");
  }
  gemm_dispatch(x, w, scales, biases, table_dtype, y, y_dtype, ro, src_row, out_row, P, T, E, N, K,
                group_size, bits, mode, st);
  return check_launch("gather gemm launch");
}

int qmm_quantized_matmul(const void* x, int x_dtype, const void* w, const void* scales,
                         const void* biases, int table_dtype, void* y, int y_dtype,
                         int64_t batch, int64_t M, int64_t N, int64_t K, int group_size,
                         int bits, int mode, void* workspace, size_t workspace_bytes,
                         void* stream) {
  const int terms = act_terms(x_dtype);
  if (batch > 0 && batch <= 65535 && M > 0 && N > 0 && K > 0 && terms * M > kGemvMaxM && x && w && scales && y) {
    const size_t xb = (size_t)M * K * (x_dtype == QMM_F32 ? 4 : 2), yb = (size_t)M * N * (y_dtype == QMM_F32 ? 4 : 2);
    const size_t wb = (size_t)N * (K * (mode == QMM_MODE_MXFP4 ? 4 : bits) / 8);
    const size_t tb = mode == QMM_MODE_MXFP4 ? (size_t)N * (K / 32) : (size_t)N * (K / std::max(group_size, 1)) * (table_dtype == QMM_F32 ? 4 : 2);
    int rc = QMM_OK;
    int64_t z = 0;
    // (what dense_bf16 and the terms below would refuse)
    const size_t inner = dense_scratch(terms * M, N, K, mode, terms > 1);
    const bool taken = workspace_bytes >= inner + (terms > 1 ? term_bytes(terms, batch * M, N, K) : 0) &&
                       (inner == 0 || aligned16(scales)) && (terms == 1 || batch * terms * M * K < (1ll << 30));
    for (; taken && z < batch; ++z)
      if (!ran_short(static_cast<const char*>(x) + z * xb, x_dtype, static_cast<const char*>(w) + z * wb,
                     static_cast<const char*>(scales) + z * tb, biases ? static_cast<const char*>(biases) + z * tb : nullptr,
                     table_dtype, static_cast<char*>(y) + z * yb, y_dtype, nullptr, nullptr, nullptr, M, M, 1, N, K,
                     group_size, bits, mode, workspace, workspace_bytes, stream, &rc) || rc)
        break;
    if (z == batch || rc) return rc;
    // (batch entries differ in their tables' alignment alone: the ones that ran are computed again below)
  }
  if (terms == 1 || batch <= 0 || M <= 0 || N <= 0 || K <= 0 || !x)
    return dense_bf16(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, batch, M, N, K,
                      group_size, bits, mode, workspace, workspace_bytes, stream, false);
  // bf16 terms as extra rows: x2 [batch, terms * M, K] -> p2 [batch, terms * M, N] -> y
  if (!aligned16(x)) return fail(QMM_ERR_BAD_ARGUMENT, "activation pointer not 16-byte aligned");
  if (batch * terms * M * K >= (1ll << 30))
    return fail(QMM_ERR_BAD_SHAPE, "shape exceeds kernel index range");
  const size_t xs = align256((size_t)(batch * terms * M * K) * 2);
  const size_t ps = align256((size_t)(batch * terms * M * N) * 4);
  const size_t inner = dense_scratch(terms * M, N, K, mode, true);
  if (!workspace || workspace_bytes < xs + ps + inner || !aligned16(workspace))
    return fail(QMM_ERR_WORKSPACE, "float16 / float32 activations need %zu aligned workspace bytes, got %zu",
                xs + ps + inner, workspace ? workspace_bytes : (size_t)0);
  char* ws = static_cast<char*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  int rc;
  if (terms * M <= kGemvMaxM && batch <= 65535 && N <= INT32_MAX && y && mode == QMM_MODE_MXFP4 &&
      (gemv_runs_general(N, K, group_size, bits, mode, table_dtype, scales, biases, batch) ? K <= kTermsCodesGeneral
                                                                                           : terms_dense(batch, N, K))) {
    // (the general MXFP4 decode kernel splits them itself)
    rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
    if (rc) return rc;
    gemv_terms_dispatch(x, x_dtype, w, scales, y, y_dtype, batch, M, N, K, nullptr, nullptr, nullptr, nullptr, nullptr,
                        0, 0, 0, st);
    return check_launch("gemv launch");
  }
  split_terms_dispatch(x, x_dtype, ws, batch, M, K, nullptr, -1, st);
  rc = check_launch("activation split launch");
  if (rc) return rc;
  rc = dense_bf16(ws, QMM_BF16, w, scales, biases, table_dtype, ws + xs, QMM_F32, batch, terms * M, N, K,
                  group_size, bits, mode, inner ? ws + xs + ps : nullptr, workspace_bytes - xs - ps, stream, true);
  if (rc) return rc;
  if (!y) return fail(QMM_ERR_BAD_ARGUMENT, "null output pointer");
  sum_terms_dispatch(ws + xs, terms, y, y_dtype, batch, M, N, nullptr, nullptr, 0, st);
  return check_launch("term sum launch");
}

// The sorted-rows product.  A kernel that clears the rows `clear` asks for on the
// way takes its y away.
static int grouped_product(const void* x, int x_dtype, const void* w, const void* scales,
                           const void* biases, int table_dtype, void* y, int y_dtype,
                           const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                           int group_size, int bits, int mode, void* workspace, size_t workspace_bytes,
                           void* stream, ClearArgs* clear) {
  const int terms = act_terms(x_dtype);
  int rs = QMM_OK;
  // (wider activations are refused without room for their terms and the terms' products)
  const bool taken = terms == 1 || (R > 0 && N > 0 && K > 0 &&
                                    workspace_bytes >= term_bytes(terms, R, N, K) + dense_scratch(R, N, K, mode, true));
  if (row_offsets && taken &&
      ran_short(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, row_offsets, nullptr, nullptr, R, R, E, N, K,
                group_size, bits, mode, workspace, workspace_bytes, stream, &rs))
    return rs;
  if (terms == 1 || R <= 0 || E <= 0 || N <= 0 || K <= 0 || !x || !row_offsets || !y)
    return grouped_bf16(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, row_offsets, R, E, N, K,
                        group_size, bits, mode, workspace, workspace_bytes, stream, false, clear);
  // one grouped product per bf16 term (the rows keep their expert order)
  if (!aligned16(x)) return fail(QMM_ERR_BAD_ARGUMENT, "activation pointer not 16-byte aligned");
  const size_t xs = align256((size_t)(terms * R * K) * 2), ps = align256((size_t)(terms * R * N) * 4);
  const size_t inner = dense_scratch(R, N, K, mode, true);
  if (!workspace || workspace_bytes < xs + ps + inner || !aligned16(workspace))
    return fail(QMM_ERR_WORKSPACE, "float16 / float32 activations need %zu aligned workspace bytes, got %zu",
                xs + ps + inner, workspace ? workspace_bytes : (size_t)0);
  char* ws = static_cast<char*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  split_terms_dispatch(x, x_dtype, ws, 1, R, K, nullptr, -1, st);
  int rc = check_launch("activation split launch");
  ClearArgs none{};
  for (int t = 0; t < terms && !rc; ++t)
    rc = grouped_bf16(ws + (size_t)t * R * K * 2, QMM_BF16, w, scales, biases, table_dtype,
                      ws + xs + (size_t)t * R * N * 4, QMM_F32, row_offsets, R, E, N, K, group_size, bits,
                      mode, inner ? ws + xs + ps : nullptr, inner, stream, true, &none);
  if (rc) return rc;
  sum_terms_dispatch(ws + xs, terms, y, y_dtype, 1, R, N, row_offsets, nullptr, E, st);
  return check_launch("term sum launch");
}

int qmm_grouped_qmm(const void* x, int x_dtype, const void* w, const void* scales,
                    const void* biases, int table_dtype, void* y, int y_dtype,
                    const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                    int group_size, int bits, int mode, void* workspace, size_t workspace_bytes,
                    void* stream) {
  ClearArgs none{};
  return grouped_product(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, row_offsets, R, E, N, K,
                         group_size, bits, mode, workspace, workspace_bytes, stream, &none);
}

int qmm_grouped_qmm_zeroed(const void* x, int x_dtype, const void* w, const void* scales,
                           const void* biases, int table_dtype, void* y, int y_dtype,
                           const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                           int group_size, int bits, int mode, void* workspace, size_t workspace_bytes,
                           void* stream) {
  const bool rows = y && row_offsets && R > 0 && R <= INT32_MAX && E >= 0 && E <= 65535 && N > 0 && N <= INT32_MAX;
  ClearArgs clear{};
  if (rows) clear = ClearArgs{y, row_offsets, (int)R, (int)E, N * (y_dtype == QMM_F32 ? 4 : 2)};
  const int rc = grouped_product(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, row_offsets, R, E, N, K,
                                 group_size, bits, mode, workspace, workspace_bytes, stream, &clear);
  if (rc || !clear.y) return rc;
  clear_rows_dispatch(clear, static_cast<hipStream_t>(stream));
  return check_launch("row clearing launch");
}

int qmm_gather_qmm(const void* x, int x_dtype, const void* w, const void* scales,
                   const void* biases, int table_dtype, void* y, int y_dtype,
                   const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t T,
                   int64_t E, int64_t N, int64_t K, int group_size, int bits, int mode,
                   void* workspace, size_t workspace_bytes, void* stream) {
  const int terms = act_terms(x_dtype);
  if (terms == 1 || P <= 0 || T < 0 || E < 0 || N <= 0 || K <= 0 || !x || !rhs_idx || !y)
    return gather_bf16(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, lhs_idx, rhs_idx, P, T, E,
                       N, K, group_size, bits, mode, workspace, workspace_bytes, stream, false);
  // More pairs than the decode kernels take: short groups read float16 / float32
  // activations as they are.  Not where the grouped decode multiplies affine weights:
  // it keeps them exact, the short-group kernel rounds them to bf16 (1e-7 against
  // 1.6e-3 from the product of the exact weights, 128 pairs over 8 experts of 1024 x
  // 4096, eight-bit codes; four-bit ones 4e-7).  MXFP4 weights are exact in both.
  const int own = short_terms(x_dtype, table_dtype, group_size, mode);
  const size_t inner = gather_scratch(P, E, N, K, true);
  // (what follows needs the workspace for more than the sort)
  const bool odd = workspace && aligned16(x) && mode == QMM_MODE_MXFP4 && sorts_odd(P, E, N, K, mode, workspace_bytes);
  const bool in_kernel = odd || terms_in_kernel(x, terms, P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, y_dtype, inner);
  const bool exact_decode = mode == QMM_MODE_AFFINE && (bits == 4 || bits == 8) && (group_size == 64 || group_size == 128) &&
                            K % group_size == 0 &&
                            grouped_decode_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, ~(size_t)0);
  if (!in_kernel && !exact_decode && P > kGatherGemvMaxPairs && P <= INT32_MAX / 2 && E > 0 && E <= 65535 && workspace && aligned16(workspace) &&
      workspace_bytes >= route_bytes(P, E) + short_prep_bytes(P, K, own) &&
      workspace_bytes >= term_bytes(terms, P, N, K) + gather_scratch(P, E, N, K, true) &&
      short_wins(P, E, N, K, bits, mode, terms, own, true, workspace_bytes - route_bytes(P, E)) &&
      short_supported(P, E, N, K, mode == QMM_MODE_MXFP4 ? 32 : std::max(group_size, 1), bits, mode, table_dtype, own, scales, biases)) {
    const size_t need = route_bytes(P, E);
    int32_t* ro = static_cast<int32_t*>(workspace);
    int32_t* cursor = ro + E + 1;
    int32_t* src_row = cursor + E;
    int32_t* out_row = src_row + P;
    int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
    if (!rc) rc = check_io(x, x_dtype, y, y_dtype);
    if (rc) return rc;
    route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, nullptr, static_cast<hipStream_t>(stream));
    rc = check_launch("route launch");
    if (rc) return rc;
    if (ran_short(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, ro, src_row, out_row, P, T, E, N, K, group_size,
                  bits, mode, static_cast<char*>(workspace) + need, workspace_bytes - need, stream, &rc))
      return rc;
  }
  // the pairs' rows are gathered while they are split; every term is then a
  // gathered product over rows already in pair order
  const size_t xs = align256((size_t)(terms * P * K) * 2), ps = align256((size_t)(terms * P * N) * 4);
  if (!workspace || workspace_bytes < xs + ps + inner || !aligned16(workspace))
    return fail(QMM_ERR_WORKSPACE, "float16 / float32 activations need %zu aligned workspace bytes, got %zu",
                xs + ps + inner, workspace ? workspace_bytes : (size_t)0);
  if (terms * P * K >= (1ll << 30)) return fail(QMM_ERR_BAD_SHAPE, "shape exceeds kernel index range");
  char* ws = static_cast<char*>(workspace);
  hipStream_t st = static_cast<hipStream_t>(stream);
  // The general MXFP4 decode kernel splits the rows itself: one launch for pairs of their
  // own, two for sorted ones.
  if (in_kernel) {
    int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
    if (!rc) rc = check_io(ws, QMM_BF16, ws + xs, QMM_F32);
    if (rc) return rc;
    if (!odd && !sorts_general(P, E, inner)) {
      gemv_terms_dispatch(x, x_dtype, w, scales, y, y_dtype, P, 1, N, K, lhs_idx, rhs_idx, nullptr, nullptr, nullptr, E, T, 0, st);
      return check_launch("gather gemv launch");
    }
    if (sorts_itself(P, E, N)) {
      gemv_terms_dispatch(x, x_dtype, w, scales, y, y_dtype, skinny2_max_segments(P, E), 16, N, K, lhs_idx, rhs_idx, nullptr,
                          nullptr, nullptr, E, T, (int)P, st);
      return check_launch("grouped gemv launch");
    }
    int32_t* ro = reinterpret_cast<int32_t*>(ws);
    int32_t* cursor = ro + E + 1;
    int32_t* src_row = cursor + E;
    int32_t* out_row = src_row + P;
    int32_t* segments = out_row + P;
    route(lhs_idx, rhs_idx, P, E, ro, cursor, src_row, out_row, segments, st);
    rc = check_launch("route launch");
    if (rc) return rc;
    gemv_terms_dispatch(x, x_dtype, w, scales, y, y_dtype, skinny2_max_segments(P, E), 16, N, K, nullptr, nullptr, segments,
                        src_row, out_row, E, T, 0, st);
    return check_launch("grouped gemv launch");
  }
  // Pairs that are decode products of their own: the terms are the rows of one (terms
  // <= 16: a pair's weight is streamed once, in one launch instead of one a term).
  // In groups of 32 fewer than sixteen pairs are, unless the experts are so few that once a
  // term each is less than once a pair (us, as rows / sorted once a term: float32, 4 pairs over 64
  // experts of 440 x 1472 10.3 / 27.6, 8 of 11880 x 2816 over 8 69 / 207, 15 of 4744 x 8768 over 4 124 / 106,
  // float16, 14 of 4160 x 8000 over 8 73 / 116, 12 of 7280 x 4160 over 4 82 / 66).
  const bool rows_win = mode == QMM_MODE_AFFINE && group_size == 32 && P < 16 && terms * E >= P;
  if (P <= kGatherGemvMaxPairs && E <= 65535 && N <= INT32_MAX && K <= INT32_MAX &&
      !sorted_here_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases) &&
      (!grouped_decode_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, inner) || rows_win) &&
      !grouped_general_serves(P, E, N, K, group_size, bits, mode, table_dtype, scales, biases, inner)) {
    int rc = check_quant(N, K, group_size, bits, mode, table_dtype, w, scales, biases);
    if (!rc) rc = check_io(ws, QMM_BF16, ws + xs, QMM_F32);
    if (rc) return rc;
    split_terms_dispatch(x, x_dtype, ws, P, 1, K, lhs_idx, T, st);    // [P, terms, K]
    rc = check_launch("activation split launch");
    if (rc) return rc;
    gemv_dispatch(ws, w, scales, biases, table_dtype, ws + xs, QMM_F32, P, terms, N, K, group_size, bits, mode, nullptr,
                  rhs_idx, E, P, st);
    rc = check_launch("gather gemv launch");
    if (rc) return rc;
    sum_terms_dispatch(ws + xs, terms, y, y_dtype, P, 1, N, nullptr, rhs_idx, E, st);
    return check_launch("term sum launch");
  }
  split_terms_dispatch(x, x_dtype, ws, 1, P, K, lhs_idx, T, st);      // lhs_idx null: row p of x
  int rc = check_launch("activation split launch");
  for (int t = 0; t < terms && !rc; ++t)
    rc = gather_bf16(ws + (size_t)t * P * K * 2, QMM_BF16, w, scales, biases, table_dtype,
                     ws + xs + (size_t)t * P * N * 4, QMM_F32, nullptr, rhs_idx, P, P, E, N, K, group_size,
                     bits, mode, inner ? ws + xs + ps : nullptr, inner, stream, true);
  if (rc) return rc;
  sum_terms_dispatch(ws + xs, terms, y, y_dtype, 1, P, N, nullptr, rhs_idx, E, st);
  return check_launch("term sum launch");
}

int qmm_gather_qmm_static(const void* x, int x_dtype, const void* w, const void* scales,
                          const void* biases, int table_dtype, void* y, int y_dtype,
                          const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t T,
                          int64_t E, int64_t N, int64_t K, int group_size, int bits, int mode,
                          void* stream) {
  if (P < 0 || T < 0 || E < 0 || N < 0 || K < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  const size_t need = gather_minimum(P, E, N, K, x_dtype);
  if (need > (size_t)QMM_STATIC_SCRATCH_BYTES)
    return fail(QMM_ERR_WORKSPACE,
                "gather_qmm_static: %lld pairs over %lld experts of [%lld, %lld] need %zu scratch "
                "bytes, the static scratch holds %zu (use qmm_gather_qmm with a workspace)",
                (long long)P, (long long)E, (long long)N, (long long)K, need,
                (size_t)QMM_STATIC_SCRATCH_BYTES);
  void* ptr = nullptr;
  if (need) {
    const int rc = static_scratch(&ptr);
    if (rc) return rc;
  }
  return qmm_gather_qmm(x, x_dtype, w, scales, biases, table_dtype, y, y_dtype, lhs_idx, rhs_idx, P,
                        T, E, N, K, group_size, bits, mode, ptr, need ? (size_t)QMM_STATIC_SCRATCH_BYTES : 0,
                        stream);
}

int qmm_dequantize(const void* w, const void* scales, const void* biases, int table_dtype,
                   void* out, int out_dtype, int64_t rows, int64_t K, int group_size, int bits,
                   int mode, void* stream) {
  if (rows < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (rows == 0 || K == 0) return QMM_OK;
  int rc = check_quant(rows, K, group_size, bits, mode, table_dtype, w, scales, biases);
  if (rc) return rc;
  if (!out) return fail(QMM_ERR_BAD_ARGUMENT, "null output pointer");
  if (out_dtype != QMM_F32 && out_dtype != QMM_BF16 && out_dtype != QMM_F16)
    return fail(QMM_ERR_UNSUPPORTED, "output dtype %d", out_dtype);
  if (!aligned16(out)) return fail(QMM_ERR_BAD_ARGUMENT, "output pointer not 16-byte aligned");
  dequant_dispatch(w, scales, biases, table_dtype, out, out_dtype, rows, K, group_size, bits,
                   mode, static_cast<hipStream_t>(stream));
  return check_launch("dequantize launch");
}

static int check_codes(const void* a, const void* b, int64_t rows, int64_t K, int bits) {
  if (rows < 0 || K < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (bits != 2 && bits != 4 && bits != 8) return fail(QMM_ERR_UNSUPPORTED, "bits=%d (2, 4 or 8)", bits);
  if (K % (32 / bits)) return fail(QMM_ERR_BAD_SHAPE, "K=%lld not a multiple of %d", (long long)K, 32 / bits);
  if (rows * K == 0) return QMM_OK;
  if (!a || !b) return fail(QMM_ERR_BAD_ARGUMENT, "null pointer");
  if (!aligned16(a) || !aligned16(b)) return fail(QMM_ERR_BAD_ARGUMENT, "pointer not 16-byte aligned");
  return QMM_OK;
}

int qmm_unpack_codes(const void* w, void* codes, int64_t rows, int64_t K, int bits, void* stream) {
  int rc = check_codes(w, codes, rows, K, bits);
  if (rc || rows * K == 0) return rc;
  unpack_dispatch(w, codes, rows, K, bits, static_cast<hipStream_t>(stream));
  return check_launch("unpack launch");
}

int qmm_pack_codes(const void* codes, void* w, int64_t rows, int64_t K, int bits, void* stream) {
  int rc = check_codes(codes, w, rows, K, bits);
  if (rc || rows * K == 0) return rc;
  pack_dispatch(codes, w, rows, K, bits, static_cast<hipStream_t>(stream));
  return check_launch("pack launch");
}

int qmm_take_k(const void* x, int x_dtype, const int32_t* perm, void* out, int64_t rows,
               int64_t K, void* stream) {
  if (rows < 0 || K < 0) return fail(QMM_ERR_BAD_ARGUMENT, "negative shape");
  if (rows * K == 0) return QMM_OK;
  if (!x || !perm || !out) return fail(QMM_ERR_BAD_ARGUMENT, "null pointer");
  if (x_dtype != QMM_F32 && x_dtype != QMM_BF16 && x_dtype != QMM_F16)
    return fail(QMM_ERR_UNSUPPORTED, "dtype %d", x_dtype);
  take_dispatch(x, x_dtype, perm, out, rows, K, static_cast<hipStream_t>(stream));
  return check_launch("take launch");
}

}  // extern "C"
