/* qmm_hip.h -- C ABI of libqmm_hip.so: quantized matmul for MI355X (gfx950).
 *
 * The library serves the fused op that the reference's quantized-matmul
 * recognizer emits.  Every entry point takes raw DEVICE pointers and explicit
 * shapes; the caller owns every buffer (including the optional workspace); no
 * entry point allocates, frees or synchronizes; work is enqueued on the given
 * HIP stream (a hipStream_t passed as void*, NULL = the default stream).
 *
 * Return value: 0 on success, else one of the QMM_ERR_* codes; the message of
 * the calling thread's last failure is available from qmm_last_error().
 * A non-zero status means nothing was launched, so a caller can run the
 * literal (unfused) chain instead, which is what the reference's handler does
 * on any exception (reference src/metaljax/qmm.py:2348-2355).
 *
 * Layouts (identical to what the reference hands mx.quantized_matmul,
 * reference src/metaljax/qmm.py:2469-2501 and :206-282):
 *   x        [batch, M, K] row-major, dtype x_dtype (bf16, or float16 / float32:
 *            those are split, exactly, into two / three bf16 terms that are
 *            multiplied like bf16 activations and added in float32 -- the
 *            workspace queries take x_dtype for that)
 *   w        affine: uint32 [batch, N, K*bits/32]; element i of a row at bits
 *            [i*bits, (i+1)*bits) of the row's little-endian stream.
 *            mxfp4:  the same stream of 4-bit E2M1 codes (uint32 [N, K/8] ==
 *            uint8 [N, K/2], low nibble = even element)
 *   scales   affine: [batch, N, K/group_size] in table_dtype;
 *            mxfp4:  uint8 E8M0 [batch, N, K/32]
 *   biases   affine: like scales; mxfp4: NULL
 *   y        [batch, M, N] row-major, dtype y_dtype
 * Semantics: y = x . dequant(w)^T with float32 accumulation, where
 *   affine  w = scales*q + biases          (one fused multiply-add)
 *   mxfp4   w = E2M1[code] * 2^(scale-127)
 */
#ifndef QMM_HIP_H_
#define QMM_HIP_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

enum {
  QMM_OK = 0,
  QMM_ERR_BAD_ARGUMENT = 1,  /* null pointer, negative size, misaligned pointer */
  QMM_ERR_BAD_SHAPE = 2,     /* K % group_size, K % 32, ... */
  QMM_ERR_UNSUPPORTED = 3,   /* a dtype / bits / group_size combination not built */
  QMM_ERR_WORKSPACE = 4,     /* workspace missing or too small */
  QMM_ERR_HIP = 5            /* a HIP runtime call failed */
};

enum { QMM_F32 = 0, QMM_BF16 = 1, QMM_F16 = 2 };
enum { QMM_MODE_AFFINE = 0, QMM_MODE_MXFP4 = 1 };

/* Which kernel family a shape is routed to (returned by qmm_plan). */
enum { QMM_KERNEL_GEMV = 1, QMM_KERNEL_GEMM = 2, QMM_KERNEL_MXFP4_MFMA = 3 };

int qmm_abi_version(void);
const char* qmm_last_error(void);

/* Replaces mx.quantized_matmul(x, w, scales, biases, transpose=True,
 * group_size, bits, mode) -- reference src/metaljax/qmm.py:2491.
 * `batch` > 1 multiplies batch independent [M,K] x [N,K] pairs (the batched
 * dot of reference src/metaljax/qmm.py:65-69).  `workspace` may be NULL when
 * qmm_workspace_bytes() returns 0 for the same arguments. */
int qmm_quantized_matmul(const void* x, int x_dtype, const void* w, const void* scales,
                         const void* biases, int table_dtype, void* y, int y_dtype,
                         int64_t batch, int64_t M, int64_t N, int64_t K, int group_size,
                         int bits, int mode, void* workspace, size_t workspace_bytes,
                         void* stream);

/* Scratch bytes qmm_quantized_matmul / qmm_grouped_qmm run best with for these
 * arguments (M = total rows for the grouped form); always enough.  The float32
 * sums of a K that is split over workgroups are part of it: a call with less
 * runs with fewer splits, and is refused (QMM_ERR_WORKSPACE) only where the
 * rest -- the re-laid activations, the terms of float16 / float32 ones and
 * their products -- does not fit.  (bf16 rows of the grouped form run with any
 * workspace, on a slower kernel.) */
size_t qmm_workspace_bytes(int64_t batch, int64_t M, int64_t N, int64_t K, int group_size,
                           int bits, int mode, int x_dtype);

/* Scratch bytes qmm_gather_qmm wants for P pairs over E experts of [N, K]
 * weights (0 below four pairs, which run as independent decode products): the
 * expert sort's arrays, plus the segment list of the grouped decode (up to
 * 16 pairs an expert on average: one decode product per expert and sixteen
 * pairs) or the re-laid activation copy of the prefill kernel (more pairs), for
 * float16 / float32 activations also their terms and the terms' products; and
 * the sums of a split K, as far as they fit QMM_STATIC_SCRATCH_BYTES.
 * With less the call still runs, on a slower kernel or with fewer splits; bf16
 * activations need the expert sort's arrays above 64 pairs, float16 and float32
 * ones everything but the sums. */
size_t qmm_gather_workspace_bytes(int64_t P, int64_t E, int64_t N, int64_t K, int x_dtype);

/* The kernel family and launch geometry the dispatcher would choose. */
int qmm_plan(int64_t M, int64_t N, int64_t K, int group_size, int bits, int mode,
             int* kernel, int* grid, int* block);

/* Replaces mx.gather_qmm(x, w, scales, biases, lhs_idx, rhs_idx, transpose=True, ...)
 * with one row per pair -- reference src/metaljax/moe.py:1320:
 *   y[p, :] = x[lhs_idx[p], :] . dequant(w[rhs_idx[p]])^T     p in [0, P)
 * x [T, K]; w/scales/biases carry a leading expert axis [E, N, ...];
 * lhs_idx, rhs_idx int32 [P] on the device, in any order; y [P, N].
 * lhs_idx may be NULL (identity). */
int qmm_gather_qmm(const void* x, int x_dtype, const void* w, const void* scales,
                   const void* biases, int table_dtype, void* y, int y_dtype,
                   const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t T,
                   int64_t E, int64_t N, int64_t K, int group_size, int bits, int mode,
                   void* workspace, size_t workspace_bytes, void* stream);

/* qmm_gather_qmm for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * No counterpart in the reference.  Same arguments and results as
 * qmm_gather_qmm without the workspace pair: the expert sort's arrays, the
 * segment list and the re-laid activation copy live in a device array of
 * QMM_STATIC_SCRATCH_BYTES that is part of the library's code object (every
 * GPU the library runs on holds one until the process ends).  A call whose
 * qmm_gather_workspace_bytes(P, E, N, K, x_dtype) exceeds that size fails with
 * QMM_ERR_WORKSPACE and launches nothing.  The call allocates and frees
 * nothing.  Every call on a GPU uses that GPU's one array: calls that overlap
 * on one GPU (different streams, or threads) race; calls in stream order do
 * not, and each call initialises what it reads.  The first call on a device
 * looks up the array's address and sets kernel attributes: make it outside a
 * stream capture (any call, of any size); later calls only launch kernels. */
#define QMM_STATIC_SCRATCH_BYTES (16u << 20)
int qmm_gather_qmm_static(const void* x, int x_dtype, const void* w, const void* scales,
                          const void* biases, int table_dtype, void* y, int y_dtype,
                          const int32_t* lhs_idx, const int32_t* rhs_idx, int64_t P, int64_t T,
                          int64_t E, int64_t N, int64_t K, int group_size, int bits, int mode,
                          void* stream);

/* The sorted-rows form of the same product (rows of x already grouped by
 * expert): rows [row_offsets[e], row_offsets[e+1]) use expert e's weight.
 * row_offsets int32 [E+1] on the device, non-decreasing, row_offsets[0] = 0,
 * row_offsets[E] = R.  Empty experts are legal.  No host synchronization.
 * Serves the per-expert product of reference src/metaljax/moe.py:1283-1340. */
int qmm_grouped_qmm(const void* x, int x_dtype, const void* w, const void* scales,
                    const void* biases, int table_dtype, void* y, int y_dtype,
                    const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                    int group_size, int bits, int mode, void* workspace,
                    size_t workspace_bytes, void* stream);

/* qmm_grouped_qmm into fresh memory: the rows of y outside the offsets, which
 * qmm_grouped_qmm leaves as they are, are set to zero.  y may hold anything.
 * Serves the per-expert product of reference src/metaljax/moe.py:1283-1340. */
int qmm_grouped_qmm_zeroed(const void* x, int x_dtype, const void* w, const void* scales,
                           const void* biases, int table_dtype, void* y, int y_dtype,
                           const int32_t* row_offsets, int64_t R, int64_t E, int64_t N, int64_t K,
                           int group_size, int bits, int mode, void* workspace,
                           size_t workspace_bytes, void* stream);

/* Replaces mx.dequantize(w, scales, biases, group_size, bits[, mode]) --
 * used by the reference's layout tests (tests/test_qmm.py:121;
 * tests/test_qmm_mxfp4.py:192).  rows = product of the leading dims; out
 * [rows, K] in out_dtype.  Bit-exact: float32 out is fma(scale, q, bias);
 * bf16 / f16 out is one round-to-nearest-even of that. */
int qmm_dequantize(const void* w, const void* scales, const void* biases, int table_dtype,
                   void* out, int out_dtype, int64_t rows, int64_t K, int group_size,
                   int bits, int mode, void* stream);

/* uint32 words [rows, K*bits/32] -> uint8 codes [rows, K]; inverse of the
 * reference's pack_codes (src/metaljax/qmm.py:206-232).  bits in {2, 4, 8}. */
int qmm_unpack_codes(const void* w, void* codes, int64_t rows, int64_t K, int bits,
                     void* stream);

/* uint8 codes [rows, K] -> uint32 words [rows, K*bits/32], masking each code
 * to `bits` -- reference pack_codes, src/metaljax/qmm.py:206-232. */
int qmm_pack_codes(const void* codes, void* w, int64_t rows, int64_t K, int bits,
                   void* stream);

/* out[r, j] = x[r, perm[j]]: the activation gather applied when a weight was
 * packed with a permuted contraction axis (mx.take(x, perm, -1), reference
 * src/metaljax/qmm.py:2486-2490).  perm int32 [K] on the device. */
int qmm_take_k(const void* x, int x_dtype, const int32_t* perm, void* out, int64_t rows,
               int64_t K, void* stream);

/* ---- the tensor work round an expert dispatch's products -----------------------
 * Short programs over float32 registers; an instruction rounds its result to `el`
 * (QMM_EL_F32: not at all).  Registers are named by number in a pair map, by their
 * first float in a row program. */
#define QMM_EL_F32 0
#define QMM_EL_BF16 1
#define QMM_EL_F16 2
#define QMM_EL_BOOL 3
#define QMM_EL_I32 4                                   /* outputs of a row program */
enum {
  QMM_OP_COPY, QMM_OP_ADD, QMM_OP_SUB, QMM_OP_MUL, QMM_OP_DIV, QMM_OP_MAX, QMM_OP_MIN, QMM_OP_POW, QMM_OP_ABS,
  QMM_OP_NEG, QMM_OP_EXP, QMM_OP_LOG, QMM_OP_LOGISTIC, QMM_OP_TANH, QMM_OP_SQRT, QMM_OP_RSQRT, QMM_OP_CEIL,
  QMM_OP_FLOOR, QMM_OP_RINT, QMM_OP_SIGN, QMM_OP_EQ, QMM_OP_NE, QMM_OP_LT, QMM_OP_LE, QMM_OP_GT, QMM_OP_GE,
  QMM_OP_AND, QMM_OP_OR, QMM_OP_XOR, QMM_OP_NOT,
  QMM_OP_SELECT,                                       /* a ? b : c */
  QMM_OP_CLAMP,                                        /* b between a and c */
  QMM_OP_IMM,
  QMM_OP_SUM, QMM_OP_ROWMAX, QMM_OP_ROWMIN,            /* row programs only, from here on */
  QMM_OP_SLICE,                                        /* n elements of a from b on, c apart */
  QMM_OP_TOPK                                          /* the n largest of a, largest first, equal ones by index: dst; indices: c */
};

#define QMM_MAP_LEAVES 8
#define QMM_MAP_CODE 40
#define QMM_MAP_REGISTERS 32
typedef struct { uint8_t op, dst, a, b, c, el; float imm; } qmm_instruction;
/* Element base + pair p * pair + its expert * expert + its token * token + the
 * output coordinates * coef of p. */
typedef struct { const void* p; int64_t base; int32_t pair, expert, token, coef[3], el; } qmm_map_leaf;
/* y[p, i] for the P selected (token, expert) pairs -- pair p is token
 * p / per_token and expert experts_of[p] -- and the i < inner elements of a pair
 * (coordinates dims[3 - rank..2]); leaf j starts in register j.  With `weights`
 * [P]: y[t, i] = sum over a token's pairs of weights[p] * (the result in sum_el). */
typedef struct {
  void* y;
  const void* weights;
  const int32_t* experts_of;
  int64_t pairs, inner, dims[3];
  int32_t per_token, experts, rank, y_el, sum_el, weights_el, leaves, instructions, registers, result;
  qmm_map_leaf leaf[QMM_MAP_LEAVES];
  qmm_instruction code[QMM_MAP_CODE];
} qmm_pair_map;

/* One pair map launch: the array operations between and behind the per-expert
 * products of a gathered dispatch (reference src/metaljax/moe.py:1425-1461).  An
 * expert index outside [0, experts) reads the nearest expert's data. */
int qmm_pair_map_run(const qmm_pair_map* map, void* stream);

/* A product of MXFP4 experts and the pair map that alone reads it, as one launch:
 * pair p multiplies row p / x_per of x [x_rows, k] by expert experts_of[p] of w
 * [experts, n, k / 8 words] with block scales s, rounded to product_el; leaf
 * col_leaf[t] of the map (whose p is null) is column col_base[t] + col_step[t] *
 * element of that.  An expert index outside [0, experts) multiplies by the nearest
 * expert, as the map reads that one's data, however the pairs are taken.  UNSUPPORTED
 * where a product and a map are the better launches (by the mode, the sizes, the types
 * and the alignment alone).  `sorted` is the library's. */
typedef struct {
  const void *x, *w, *s;
  int64_t x_rows, n, k, mode;
  int32_t x_el, x_per, product_el, tiles, col_leaf[2], col_base[2], col_step[2], sorted;
  qmm_pair_map map;
} qmm_pair_product;

/* One pair product launch (the per-expert product of reference
 * src/metaljax/moe.py:1283-1340 and what follows it there, :1425-1461). */
int qmm_pair_product_run(const qmm_pair_product* product, void* stream);

#define QMM_ROW_LEAVES 8
#define QMM_ROW_CODE 48
#define QMM_ROW_OUTS 2
#define QMM_ROW_FLOATS 8192
typedef struct { int32_t op, el, dst, n, a, an, b, bn, c, cn; float imm; } qmm_row_instruction;
typedef struct { const void* p; int64_t base, token, step; int32_t el, dst, n; } qmm_row_leaf;
typedef struct { void* p; int32_t el, src, srcn, n; } qmm_row_out;
/* For every token: optionally a row of a product (dot_x[t] . dot_w, dot_n columns
 * over dot_k, float32 sums; dot_cols: dot_n rounded up to a power of two) into
 * register dot_dst, then the leaves, then the program; out[j] is [tokens, n]. */
typedef struct {
  const void *dot_x, *dot_w;
  int64_t dot_x_t, dot_x_k, dot_w_n, dot_w_k, dot_k;
  int32_t dot_n, dot_cols, dot_dst, dot_x_el, dot_w_el, dot_el;
  int32_t tokens, reg_floats, leaves, instructions, outs;
  qmm_row_leaf leaf[QMM_ROW_LEAVES];
  qmm_row_out out[QMM_ROW_OUTS];
  qmm_row_instruction code[QMM_ROW_CODE];
} qmm_row_program;

/* One row program launch: a router from its logits to the selected experts and
 * their weights (the graph of reference src/metaljax/moe.py:335-442). */
int qmm_row_program_run(const qmm_row_program* program, void* stream);

/* The arguments of qmm_gather_qmm. */
typedef struct {
  const void *x, *w, *scales, *biases;
  void* y;
  const int32_t *lhs_idx, *rhs_idx;
  void* workspace;
  int64_t workspace_bytes, table_dtype, group_size, bits, mode, pairs, rows, experts, n, k;
  int32_t x_dtype, y_dtype;
} qmm_pair_gather;

/* A call of a compiled dispatch, launch after launch: step i's program, with the
 * eight bytes at every patch's `at` replaced by values[value] + add, goes to the
 * entry point that its kind names.  A pair product that is served skips the `skip`
 * steps behind it, the launches it stands for; one that is not is passed over.  (The
 * experts of the pairs are inside the weight, as a top-k's are: qmm_gather_qmm leaves
 * the row of any other pair alone, where a pair product reads the nearest expert.)  The
 * programs are only read: several threads may run the same steps.  Stands for the
 * host side of reference src/metaljax/moe.py:1425-1461. */
enum { QMM_STEP_ROWS, QMM_STEP_PAIR_PRODUCT, QMM_STEP_MAP, QMM_STEP_GATHER };
typedef struct { int32_t at, value; int64_t add; } qmm_patch;
typedef struct {
  int32_t kind, bytes, patches, skip;
  const void* program;
  const qmm_patch* patch;
} qmm_step;
int qmm_steps_run(const qmm_step* steps, int64_t n, const uint64_t* values, int64_t n_values, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* QMM_HIP_H_ */
