/* C ABI of libmase_hip.so, continued: products that quantise their operands on the way in (conventions: mase_hip.h). */
#ifndef MASE_HIP_SCORES_H
#define MASE_HIP_SCORES_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * `batches` products with a short contraction (K <= 128) whose operands are quantised on the way in: y_b[M,N] =
 * Q(A_b)[M,K] * W_b[N,K]^T, bfloat16 in and out, fp32 accumulation.  Q is the MXFP quantise-dequantise of mase_hip_qdq_mxfp in
 * blocks of 32 along K, element format (a_exp_bits, a_frac_bits), finite, rounded to nearest; a_exp_bits = 0: A as it is.
 * quantise_w != 0: W goes through the same Q; 0: W as it is (quantised before, or dense).  Strides in ELEMENTS between products, as for
 * mase_hip_mxfp_gemm_batched (0 shares A or W), multiples of 8.  N must be a multiple of 8, K of 32; operands 16-byte aligned.
 * The same values as quantising first and multiplying the results, up to the order of the fp32 additions.
 * Replaces the two casts and the torch.matmul of mxfp_matmul
 *   src/mase_triton/mxfp/functional/matmul.py:24-35
 * for the products of queries and keys (test/test_mxfp_functional.py:229-230).
 */
int mase_hip_mxfp_scores(const void* a, int a_exp_bits, int a_frac_bits, const void* w, int quantise_w, void* y, int64_t M,
                         int64_t N, int64_t K, int64_t batches, int64_t a_batch_stride, int64_t w_batch_stride,
                         int64_t y_batch_stride, void* stream);

/*
 * The way that is fastest for such a product (M, N, K, batches as above): 2: mase_hip_mxfp_scores with quantise_w, 1: W through
 * mase_hip_qdq_mxfp first, 0: neither (mase_hip_extract_mxfp of W, mase_hip_qdq_mxfp of A, mase_hip_mxfp_gemm_batched; also for shapes
 * that mase_hip_mxfp_scores refuses).  one_format != 0: A and W are quantised in the same format (else never 2).  Depends on its
 * arguments only.
 */
int mase_hip_mxfp_scores_plan(int64_t M, int64_t N, int64_t K, int64_t batches, int one_format);

#ifdef __cplusplus
}
#endif
#endif
