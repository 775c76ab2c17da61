// C-ABI entry point of the products with a short contraction that quantise on the way in; the kernel is in gemm_scores.h.
#include "../../include/mase_hip_scores.h"
#include "gemm_scores.h"

using namespace mase;

extern "C" int mase_hip_mxfp_scores(const void* a, int a_exp_bits, int a_frac_bits, const void* w, int quantise_w, void* y, int64_t M, int64_t N,
                                    int64_t K, int64_t batches, int64_t a_batch_stride, int64_t w_batch_stride, int64_t y_batch_stride,
                                    void* stream) {
    if (M < 0 || N < 1 || K < 1) return fail(ERR_INVALID, "M must not be negative, N and K must be positive");
    if (M == 0) return OK;   // no rows of A: nothing to compute
    if (K % 32 != 0) return fail(ERR_INVALID, "K must be a multiple of the block size");
    if (K > SCO_MAX_K || N % 8 != 0) return fail(ERR_UNSUPPORTED, "this product takes K up to 128 and N a multiple of 8");
    if (M > 0x7FFFFFFF - SCO_M || N > (1 << 23)) return fail(ERR_UNSUPPORTED, "M must fit in 31 bits and N in 23");
    if (!a || !w || !y) return fail(ERR_INVALID, "null pointer");
    if (!aligned(a, 16) || !aligned(w, 16) || !aligned(y, 16)) return fail(ERR_INVALID, "operands must be 16-byte aligned");
    if (batches < 1 || batches > 0x7FFFFFFF) return fail(ERR_INVALID, "batches must be between 1 and 2^31 - 1");
    if (a_exp_bits == 0 && quantise_w) return fail(ERR_INVALID, "W is quantised in A's format: give one");
    if (batches > 1) {
        if (a_batch_stride != 0 && a_batch_stride < M * K) return fail(ERR_INVALID, "a_batch_stride must be 0 (A shared by every product) or at least M * K");
        if (w_batch_stride != 0 && w_batch_stride < N * K) return fail(ERR_INVALID, "w_batch_stride must be 0 (W shared by every product) or at least N * K");
        if (y_batch_stride < M * N) return fail(ERR_INVALID, "y_batch_stride must be at least M * N");
        if (a_batch_stride % 8 != 0 || w_batch_stride % 8 != 0 || y_batch_stride % 8 != 0) return fail(ERR_INVALID, "batch strides must be multiples of 8");
    }
    const ScoresArgs p{static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(w), static_cast<uint16_t*>(y), (int)M, (int)N, (int)K, 0, 0, 0, 0,
                       a_batch_stride, w_batch_stride, y_batch_stride};
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (a_exp_bits == 0) return launch_scores<SFmt<4, 3>, false, false>(p, (int)batches, s);
    return dispatch_fmt(a_exp_bits, a_frac_bits, 1, RN, [&](auto f) {
        if constexpr (decltype(f)::kStatic)
            return quantise_w ? launch_scores<decltype(f), true, true>(p, (int)batches, s) : launch_scores<decltype(f), true, false>(p, (int)batches, s);
        return fail(ERR_INVALID, "MXFP element (exp_bits, frac_bits) must be one of (4,3) (5,2) (2,3) (3,2) (2,1)");
    });
}
