/*
 * ttlinear — the linear layer y = x . w^T + bias for MI355X (gfx950) behind a plain C ABI, in the same library as
 * ttsdpa (libttsdpa.so): the projections on either side of attention (QKV, output, MLP).
 *
 * Replaces, for this call shape, the reference's op::matmul(input, weight, false, true, bias) behind
 * function::linear (reference src/Function/FuncNNLayer.h:14-19, 270-272; host side src/Operation/OpLinalg.cpp:244-276;
 * its device GEMM is a cuBLAS call, src/Operation/OpLinalgCuda.cuh:239-293; CPU loop src/Operation/OpLinalgCpu.h:119-150).
 * The op implementation passes raw device pointers, sizes, leading dimensions and its current stream.
 */
#ifndef TTLINEAR_H_
#define TTLINEAR_H_

#include <stddef.h>
#include <stdint.h>

#include "ttsdpa.h"

#ifdef __cplusplus
extern "C" {
#endif

enum ttlinear_route {
  TTLINEAR_ROUTE_NONE = 0,   /* empty output */
  TTLINEAR_ROUTE_MFMA = 1,   /* K a multiple of 64 (fp16/bf16) or 32 (fp32), 16-byte aligned rows, N a multiple of 4:
                                a matrix-core kernel reads the operands as they lie, fp32 accumulation (fp32 tensors: full fp32 products) */
  TTLINEAR_ROUTE_GENERAL = 2 /* everything else (other K, unaligned rows): the streaming MFMA kernel, which takes any alignment, or, given
                                scratch (ttlinear_matmul), the tiled ones on copies in whole k-tiles where that is faster; the vector
                                ALUs only for contraction-major operands of fewer than 16 rows and for empty contractions */
};

/* out[m, n] = bias[n] + sum_k x[m, k] * w[n, k]   (m < M, n < N, k < K)
 * x: [M, K] with row stride ldx elements; w: [N, K] (the layout of a Linear layer's weight) with row stride ldw;
 * bias: [N] or NULL; out: [M, N] with row stride ldo.  dtype is a ttsdpa_dtype shared by all four tensors.
 * Accumulation is fp32 starting from the bias (the reference writes the bias into C and accumulates onto it), one
 * rounding to the element type at the end.  K == 0 yields the bias (or zeros).
 * Enqueues on `stream` (a hipStream_t; NULL = the default stream); no allocation, no synchronisation.
 * Returns a ttsdpa_status code, or a positive hipError_t. */
int ttlinear_forward(int dtype, const void* x, const void* w, const void* bias, void* out, int64_t M, int64_t N,
                     int64_t K, int64_t ldx, int64_t ldw, int64_t ldo, void* stream);

/* Validate the arguments and report the kernel ttlinear_forward would pick (enum ttlinear_route).  Launches nothing. */
int ttlinear_plan(int dtype, const void* x, const void* w, const void* bias, const void* out, int64_t M, int64_t N,
                  int64_t K, int64_t ldx, int64_t ldw, int64_t ldo, int* route);

/* out[m, n] = bias[n] + sum_k A(m, k) * B(k, n) with the reference's transpose flags — op::matmul(a, b, transA, transB,
 * bias) for 2-D operands (reference src/Operation/OpLinalgCpu.h:119-150: a is [M, K], or [K, M] with transA; b is [K, N], or
 * [N, K] with transB).  (false, true) is ttlinear_forward; FuncLinear::backward (reference
 * src/Function/FuncNNLayer.h:20-33) uses the other two that matter: (false, false) for the input gradient
 * dy[M, N] . w[N, K], and (true, false) for the weight gradient dy^T . x.  lda / ldb / ldo are row strides in elements.
 * workspace: ttlinear_matmul_workspace_bytes() bytes of device scratch, 256-byte aligned (0 bytes: none is used).  Operands whose
 * layout the tiled matrix-core kernels do not take (contraction-major, rows that are not whole k-tiles, unaligned rows) are
 * copied there where product and copies together are faster than reading them in place, and products with few tiles divide
 * their contraction among workgroups ((false, true) included: what ttlinear_forward cannot do).  With less (or NULL) the
 * operands are read in place: 16-bit contraction-major ones by the tiled kernels (K a multiple of 64, N a multiple of 4,
 * 16-byte aligned operands with leading dimensions that are multiples of 8, a contraction-major operand's row count a
 * multiple of 8), others by the streaming kernel.  Same return codes as ttlinear_forward. */
size_t ttlinear_matmul_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b);
int ttlinear_matmul(int dtype, const void* a, const void* b, const void* bias, void* out, int64_t M, int64_t N, int64_t K,
                    int trans_a, int trans_b, int64_t lda, int64_t ldb, int64_t ldo, void* workspace,
                    size_t workspace_bytes, void* stream);

/* The output tiles that ttlinear_matmul makes a 16-bit product of dense, aligned operands on, given its workspace (rows x columns; OTHER:
 * fp32, the streaming kernel, operands read contraction-major).  Estimates decide: the answer may change with the library. */
enum ttlinear_tiles {
  TTLINEAR_TILES_OTHER = 0,
  TTLINEAR_TILES_128x128 = 1,
  TTLINEAR_TILES_256x256 = 2,
  TTLINEAR_TILES_128x256 = 3, /* where 256 x 256 would leave CUs idle */
  TTLINEAR_TILES_MIXED = 4    /* whole rounds of 256 x 256, what is left as 128 x 256 */
};
int ttlinear_matmul_tiles(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b);

/* The kernel and the tiles that a product of dense, aligned operands runs on, given its workspace.  Launches nothing and needs no GPU;
 * as above the answer may change with the library. */
enum ttlinear_way {
  TTLINEAR_WAY_GENERAL = 0,  /* the vector ALUs */
  TTLINEAR_WAY_STREAM = 1,   /* small tiles whose wavefronts divide the contraction among themselves */
  TTLINEAR_WAY_IN_PLACE = 2, /* large tiles of contraction-major operands read as they lie */
  TTLINEAR_WAY_TILED = 3,    /* large tiles, of copies where the layout asks for them */
  TTLINEAR_WAY_OUTER = 4     /* 128 x 128 tiles of a short contraction, both operands contraction-major */
};
typedef struct ttlinear_kernel_info {
  int32_t way;                      /* enum ttlinear_way */
  int32_t tile_rows, tile_columns;  /* STREAM: rows and columns of the output in a tile; 0 otherwise (ttlinear_matmul_tiles) */
  int32_t tiles_per_workgroup;      /* STREAM; 1 otherwise */
  int32_t shares;                   /* workgroups among which a tile's contraction is divided */
} ttlinear_kernel_info;
int ttlinear_matmul_kernel(int dtype, int64_t M, int64_t N, int64_t K, int trans_a, int trans_b, ttlinear_kernel_info* info);
/* The same of ttlinear_backward's two products, and whether they run in one launch. */
int ttlinear_backward_kernels(int dtype, int64_t M, int64_t N, int64_t K, int with_bias, ttlinear_kernel_info* of_weight,
                              ttlinear_kernel_info* of_input, int* one_launch);

/* FuncLinear::backward (reference src/Function/FuncNNLayer.h:20-33) in one call: from the upstream gradient grad [M,N], the
 * forward's x [M,K] and w [N,K] (row strides ldg, ldx, ldw in elements)
 *   grad_x [M,K] = grad . w,   grad_w [N,K] = grad^T . x,   grad_b [N] = column sums of grad (NULL: not wanted),
 * all dense, sums in fp32, one rounding of each result.  M, N, K > 0.  workspace: ttlinear_backward_workspace_bytes() bytes of
 * device scratch, 256-byte aligned.  Much of it may be for copies of the operands, which are faster to multiply than operands read
 * in place (bf16, 8192 x 6144 x 4096: 169 MB, the weight's gradient 340 us with its copies, 443 without).  With less the call
 * runs without what does not fit, down to the column sums' parts, ttlinear_backward_least_workspace_bytes() (196 KB there);
 * TTSDPA_ERR_WORKSPACE with less than that.  Enqueues on `stream`. */
size_t ttlinear_backward_least_workspace_bytes(int dtype, int64_t M, int64_t N);
size_t ttlinear_backward_workspace_bytes(int dtype, int64_t M, int64_t N, int64_t K);
int ttlinear_backward(int dtype, const void* grad, const void* x, const void* w, void* grad_x, void* grad_w, void* grad_b, int64_t M,
                      int64_t N, int64_t K, int64_t ldg, int64_t ldx, int64_t ldw, void* workspace, size_t workspace_bytes,
                      void* stream);

/* op::matmul with batch dimensions (reference src/Operation/OpLinalg.cpp:107-223: leading dimensions of the two
 * operands broadcast against each other; its device path is a strided-batched or pointer-array GEMM, its CPU path a
 * loop over the batch with per-operand offsets, :205-223).  The batch is described as up to TTLINEAR_MAX_BATCH_DIMS
 * dimensions batch_shape[0..nbatch_dims) with element strides a_batch_stride[d] / b_batch_stride[d] (0 broadcasts the
 * operand along d); batch entry i of the output, numbered row-major over batch_shape, starts at out + i * out_batch_stride.
 * Every batch entry is one ttlinear_matmul of the same M, N, K, flags and leading dimensions, enqueued in order on
 * `stream`; the workspace (ttlinear_matmul_workspace_bytes of one entry) is shared by the entries.  bias ([N] or NULL)
 * joins every entry. */
#define TTLINEAR_MAX_BATCH_DIMS 8
int ttlinear_matmul_batched(int dtype, const void* a, const void* b, const void* bias, void* out, int64_t M, int64_t N,
                            int64_t K, int trans_a, int trans_b, int64_t lda, int64_t ldb, int64_t ldo, int nbatch_dims,
                            const int64_t* batch_shape, const int64_t* a_batch_stride, const int64_t* b_batch_stride,
                            int64_t out_batch_stride, void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* TTLINEAR_H_ */
