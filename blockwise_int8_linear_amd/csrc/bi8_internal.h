// Entry points of libbi8.so for this package's own torch binding (bi8_torch.cpp); callers of the library use include/bi8.h.
// They differ from the public ones in what they leave to the caller: operands are checked there, and a contraction dimension can
// be written padded with zero codes and zero scales to the multiple of 128 that the tiled GEMM kernels want.
#pragma once

#include <stdint.h>

#include "bi8.h"

#ifdef __cplusplus
extern "C" {
#endif

/* One matrix for bi8x_quantize_dual: x [R,C] -> q [R,Cp] with scales [ceil(Cp/block), R], and qT [C,Rp] with scalesT
 * [ceil(Rp/block), C].  Rp >= R and Cp >= C: codes and scales past the matrix are written as zeros. */
typedef struct {
    const void *x;
    int8_t *q, *qT;
    float *scales, *scalesT;
    int64_t R, C, ldx, ldq, ldqt, Rp, Cp;
} Bi8DualTask;

/* `count` = 1 or 2 matrices of one type in one launch; block 32, 64 or 128, ldqt a multiple of 16 and qT 16-byte aligned
 * (BI8_ERR_UNSUPPORTED otherwise).  colsum_part (one matrix only): column sums per 128 rows, [ceil(R/128), C], for bi8x_colsum_finish. */
int bi8x_quantize_dual(const Bi8DualTask *task, int count, int x_dtype, int block, float *colsum_part, void *stream);
int bi8x_colsum_finish(const float *part, void *out, int dtype, int64_t R, int64_t C, void *stream);

/* bi8_quantize_rowwise with rows written up to column Kp >= K; Kp > K for blocks that are a power of two up to 512 (fp32: 256) and
 * x aligned to its elements (BI8_ERR_UNSUPPORTED otherwise). */
int bi8x_quantize_rowwise(const void *x, int x_dtype, int8_t *q, float *scales, int64_t M, int64_t K, int64_t Kp, int64_t ldx,
                          int64_t ldq, int block, void *stream);

/* bi8_gemm_nt_dequant_ws for a contraction that only A is padded for: K a multiple of 128 (A's codes and scales are zeros from kw
 * on), W's rows hold kw > K - 128 codes and ceil(kw/block) rows of scales.  kw < K: a multiple of 16,
 * blocks 64 and 128, 16-byte aligned rows. */
int bi8x_gemm(const int8_t *A, const int8_t *W, const float *sA, const float *sW, const void *bias, int bias_dtype, void *C, int c_dtype,
              int64_t M, int64_t N, int64_t K, int64_t kw, int64_t lda, int64_t ldw, int64_t ldc, int block, void *workspace,
              int64_t workspace_bytes, void *stream);

/* One problem of bi8x_gemm_pair: what bi8x_gemm takes, without a bias. */
typedef struct {
    const int8_t *A, *W;
    const float *sA, *sW;
    void *C;
    int64_t M, N, K, kw, lda, ldw, ldc;
} Bi8Gemm;
/* The last step of column sums (bi8x_colsum_finish) as part of a launch that follows the quantizer: part [ceil(R/128), C] -> out [C] of type dtype. */
typedef struct {
    const float *part;
    void *out;
    int dtype;
    int64_t R, C;
} Bi8ColSums;
/* Both problems in one launch where that is expected to be faster than two (BI8_ERR_UNSUPPORTED otherwise: nothing is launched); outputs of type
 * c_dtype, operands as for bi8x_gemm with rows on 16-byte boundaries, blocks 64 and 128, no scratch memory; sums: in the same launch, or NULL.  _name: the kernel whose
 * tiles the launch runs, "" where there would be none. */
int bi8x_gemm_pair(const Bi8Gemm *q, int c_dtype, int block, const Bi8ColSums *sums, void *stream);
const char *bi8x_gemm_pair_name(const Bi8Gemm *q, int c_dtype, int block);
/* bi8x_gemm without a bias, and the column sums: in the GEMM's launches where one of its kernels takes them, else in one of their own. */
int bi8x_gemm_sums(const Bi8Gemm *q, int c_dtype, int block, void *workspace, int64_t workspace_bytes, const Bi8ColSums *sums, void *stream);

/* y [M,N] = x [M,K] @ W.T + bias for 3 to 16 rows in one launch: x of C's type is quantized by the workgroups that multiply with it, the
 * bits of y are those of bi8_quantize_rowwise and bi8_gemm_nt_dequant_ws.  W, sW: codes and scales; blocks 64 and 128, K a multiple of
 * 128, x and W with 16-byte aligned rows, and up to 16 Ki activations (fp32: 8 Ki; BI8_ERR_UNSUPPORTED otherwise). */
int bi8x_linear_rows(const void *x, int dtype, const int8_t *W, const float *sW, const void *bias, int bias_dtype, void *C, int64_t M,
                     int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldc, int block, void *stream);

#ifdef __cplusplus
}
#endif
