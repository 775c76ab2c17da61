// The short-contraction kernel for the five weight formats (a translation unit of its own: the formats' other kernels take
// minutes to compile).
#include "gemm_impl.h"
#include "gemm_short_k.h"

int mase::gemm_short_k(const GemmArgs& g, int w_exp_bits, int w_frac_bits) {
    return dispatch_fmt(w_exp_bits, w_frac_bits, 1, RN, [&](auto f) {
        if constexpr (decltype(f)::kStatic) {
            return dispatch_dtype(g.out_dtype, [&](auto dt) { return launch_gemm_short_k<decltype(f), decltype(dt)::value>(g); });
        }
        return fail(ERR_INVALID, "MXFP element (exp_bits, frac_bits) must be one of (4,3) (5,2) (2,3) (3,2) (2,1)");
    });
}
