/* C ABI of libmase_hip.so, continued: linears of few rows in one launch, and weights packed at their own width (conventions: mase_hip.h). */
#ifndef MASE_HIP_LINEAR_H
#define MASE_HIP_LINEAR_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/*
 * mase_hip_mxfp_linear_scaled for a few rows in ONE launch, bfloat16 in and out: every workgroup quantises x on the way in, no scratch.  Takes
 * K % 256 = 0, 512 <= K <= 16384, N % 8 = 0 and up to 16 rows; -2 for other shapes.  Operands 16-byte aligned, w_scales 4-byte.  The
 * codes of x are those of the operand kernels; mase_hip_mxfp_linear_scaled takes this way itself where it is the faster one, which
 * mase_hip_mxfp_linear_few_plan tells (1) from the shape and the device's compute units.
 */
int mase_hip_mxfp_linear_few_plan(int64_t M, int64_t N, int64_t K);
int mase_hip_mxfp_linear_few(const void* x, int x_exp_bits, int x_frac_bits, int x_is_minifloat, const uint8_t* w_codes,
                             const uint32_t* w_scales, const void* bias, int bias_dtype, void* y, int64_t M, int64_t N, int64_t K,
                             void* stream);

/*
 * A weight of 4- or 6-bit codes (element formats (2,1), (2,3), (3,2)) packed at its own width for the block-scaled matrix instruction, which reads
 * these formats as they are: [rows_pad / 16][K / 128] tiles of 16 rows x 128 k, in a tile 64 x 16 bytes (lane 16 g + r: codes 32 g .. of row
 * r, code i at bits 4 i, or at bits 6 i with the last 8 bytes of every lane behind all first 16), rows padded to a multiple of 256;
 * scales as in the prepared form.  N a multiple of 8, K of 256 and at least 512.  mase_hip_packed_weight_bytes: size of the codes, 0 for
 * what is not packed.  A layer keeps this beside its components, as it does the prepared form.
 */
int64_t mase_hip_packed_weight_bytes(int64_t N, int64_t K, int exp_bits, int frac_bits);
int mase_hip_packed_weight_from_mxfp(const uint8_t* scales, const uint8_t* elements, int exp_bits, int frac_bits, int64_t N, int64_t K,
                                     uint8_t* out_codes, uint32_t* out_scales, void* stream);

/*
 * Products with a packed weight, bfloat16 out: A an operand (mase_hip_mxfp_gemm_packed_ws; workspace as for mase_hip_mxfp_gemm_scaled_ws, without it K is
 * not split) or bfloat16 x (mase_hip_mxfp_linear_packed; scratch 256-byte aligned, mase_hip_mxfp_linear_packed_scratch_bytes of it, none where that
 * is 0).  The values of the products with the prepared form, up to the order of the additions.  mase_hip_mxfp_packed_plan: 1 where the packed
 * weight is the faster form for M rows, by shape and format.
 */
int mase_hip_mxfp_packed_plan(int64_t M, int64_t N, int64_t K, int w_exp_bits, int w_frac_bits);
int64_t mase_hip_mxfp_gemm_packed_workspace_bytes(int64_t M, int64_t N, int64_t K, int w_exp_bits, int w_frac_bits);
int mase_hip_mxfp_gemm_packed_ws(const uint8_t* a_codes, const uint32_t* a_scales, const uint8_t* w_codes, const uint32_t* w_scales,
                                 int w_exp_bits, int w_frac_bits, const void* bias, int bias_dtype, void* y, int64_t M, int64_t N,
                                 int64_t K, void* workspace, int64_t workspace_bytes, void* stream);
int64_t mase_hip_mxfp_linear_packed_scratch_bytes(int64_t M, int64_t N, int64_t K, int w_exp_bits, int w_frac_bits);
int mase_hip_mxfp_linear_packed(const void* x, int x_exp_bits, int x_frac_bits, int x_is_minifloat, const uint8_t* w_codes,
                                const uint32_t* w_scales, int w_exp_bits, int w_frac_bits, const void* bias, int bias_dtype, void* y,
                                int64_t M, int64_t N, int64_t K, void* scratch, int64_t scratch_bytes, void* stream);

/*
 * Weight-only products of a few rows with a packed weight: A dense bfloat16 [M, K], used as it is, W composed to bfloat16 (exactly as
 * mase_hip_compose_mxfp does), products on the bf16 matrix instruction summed in fp32, bfloat16 out.  Up to 32 rows, N and K as for the packed
 * weight, K up to 65536 (16 rows) or 32768; workspace of mase_hip_mxfp_packed_dense_workspace_bytes, none where that is 0; -2 for other shapes.
 * mase_hip_mxfp_packed_dense_plan: 1 where this is faster than mase_hip_mxfp_gemm on the components, by shape and format.
 */
int mase_hip_mxfp_packed_dense_plan(int64_t M, int64_t N, int64_t K, int w_exp_bits, int w_frac_bits);
int64_t mase_hip_mxfp_packed_dense_workspace_bytes(int64_t M, int64_t N, int64_t K);
int mase_hip_mxfp_gemm_packed_dense(const void* a, const uint8_t* w_codes, const uint32_t* w_scales, int w_exp_bits, int w_frac_bits,
                                    const void* bias, int bias_dtype, void* y, int64_t M, int64_t N, int64_t K, void* workspace,
                                    int64_t workspace_bytes, void* stream);

/*
 * mase_hip_mxfp_gemm_batched for contiguous operands (strides M * K, N * K and M * N), bfloat16 A, blocks of 32, whose outputs need not be
 * 16-byte aligned from product to product: M * N of any size.
 */
int mase_hip_mxfp_matmul_batched(const void* a_dense, const uint8_t* w_scales, const uint8_t* w_elements, int w_exp_bits, int w_frac_bits,
                                 void* y, int out_dtype, int64_t M, int64_t N, int64_t K, int64_t batches, void* stream);

/*
 * `batches` products of bfloat16 x [M, K] against components in [N, K] order, lying as in mase_hip_mxfp_matmul_batched, where x is quantised to W's
 * format (blocks of 32 along K, round to nearest) on its way in: what mase_hip_qdq_mxfp and mase_hip_mxfp_matmul_batched compute, in one launch.
 * N <= 128, K % 32 == 0, bfloat16 outputs of any alignment (with N % 16 == 0, M * N a multiple of 8).
 * mase_hip_mxfp_matmul_cast_plan: 1 where this is faster than the two.
 */
int mase_hip_mxfp_matmul_cast_plan(int64_t M, int64_t N, int64_t K);
int mase_hip_mxfp_matmul_cast(const void* x, const uint8_t* w_scales, const uint8_t* w_elements, int exp_bits, int frac_bits, void* y, int64_t M, int64_t N,
                              int64_t K, int64_t batches, void* stream);

/*
 * mase_hip_mxfp_gemm_prepared_w with a workspace: products of few tiles and a long K run in several shares of K, whose fp32 sums lie in the
 * workspace (16-byte aligned, at least the bytes that the query names for this shape; 0: one share, no workspace).  With less than that, or
 * none, the product runs in one share.
 * mase_hip_mxfp_prepared_w_pays: 1 where this is faster than mase_hip_mxfp_gemm_ws on the components of the weight, 0 where it is not or where the
 * prepared form does not take the shape.
 */
int64_t mase_hip_mxfp_gemm_prepared_w_workspace_bytes(int64_t M, int64_t N, int64_t K);
int mase_hip_mxfp_gemm_prepared_w_ws(const void* a_dense, int a_dtype, const uint8_t* w_codes, const uint32_t* w_scales, const void* bias,
                                     int bias_dtype, void* y, int out_dtype, int64_t M, int64_t N, int64_t K, void* workspace,
                                     int64_t workspace_bytes, void* stream);
int mase_hip_mxfp_prepared_w_pays(int64_t M, int64_t N, int64_t K);

/*
 * For callers that build a prepared or packed weight on one stream and read it on others: has all that `stream` was given run, or what `event` (a hipEvent_t that was
 * recorded on it; or NULL) is behind?  1: yes, 0: not yet, or not to be known (a stream that is captured itself).  May be asked while other streams are captured, by
 * this thread or another; no capture is touched.
 */
int mase_hip_stream_done(void* stream, void* event);

#ifdef __cplusplus
}
#endif
#endif
