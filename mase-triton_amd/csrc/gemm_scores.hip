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

// Which way a product of short contraction goes.  The general route is a pass over each operand and the kernels that compose codes
// (gemm_short_k.h, a weight-streaming one for few rows).  GPU time in us on other operands each call, general / W in a pass before / W
// inside:
//   K = 96 pays for 128 (zeros), without the L2 prefetch of W.  Many outputs, more than one panel: 23 of 2048 x 513 27 / 31 / 37, 10 of 8192 x
//   640 41 / 45 / 53, 12 of 2048 x 384 18.6 / 24 / 24; few outputs 11.3 / 9.9 / 9.6 (one of 2048 x 1000); rows of y off the 128-byte lines or
//   short ones 58 / 42 (50 of 1000 x 1000), 60 / 51 (136 x 200 x 2048 down to 64 columns); one panel 54 / 45 inside (473 of 512 x 128), but 76 / 92 / 95
//   where rows of y are a few lines (2507 of 200 x 16);
//   K = 128, long rows of whole lines, three to twelve panels: 6 of 2048 x 768 18.6 / 24 / 24, 65536 x 768 35 / 50 / 51; outside that 64.0 / 41.7 (25 of 1000 x
//   2048), 44.6 / 40.4 (7 of 2048 x 4096);
//   K <= 64: inside up to twelve panels (2 of 8192 x 1464 19.1 / 21.9 / 18.5), before beyond that (54 / 34 with 27 of 1000 x 2048 x 64).
// A dense A, or formats that differ, rules "inside" out, and a pass over W writes twice the bytes of its codes.  Dense A, general / before: 26.1 /
// 33.4 (99 of 512 x 1000 x 64), 22.5 / 34.8 (360 of 512 x 1), 61.7 / 69.6 (32 of 2048 x 2048 x 128); 0.6 - 0.9 of the time with many rows off the lines,
// and with few outputs, where both are bound by their launches.
extern "C" int mase_hip_mxfp_scores_plan(int64_t M, int64_t N, int64_t K, int64_t batches, int one_format) {
    if (M < 1 || N < 1 || K < 1 || batches < 1 || K % 32 != 0 || K > SCO_MAX_K || N % 8 != 0 || N > (1 << 23) || M > 0x7FFFFFFF - SCO_M) return 0;
    const int64_t panels = (M + SCO_M - 1) / SCO_M;
    const double y_mb = (double)batches * (double)M * (double)N * 2e-6, w_mb = (double)batches * (double)N * (double)K * 2e-6;
    const bool few = y_mb < 9.0, many = y_mb >= 48.0, lines = N % 64 == 0;
    if (!one_format) return (few && w_mb < 9.0) || (many && !lines && panels > 2) ? 1 : 0;
    if (few) return 2;
    if (K == 96 && panels > 1) return many && panels > 2 && (!lines || N <= 512) ? 1 : 0;
    if (K == 96 && N <= 256) return 0;
    if (K == 128 && lines && N >= 2048 && panels > 2 && panels <= 12) return 0;
    return panels * (K <= 64 ? 64 : 128) <= (K <= 64 ? 768 : 512) ? 2 : 1;
}
