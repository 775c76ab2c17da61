// Test helpers, not part of the product's C ABI: which kernel a launcher picks for a shape, so that a test can say which one it means to
// run and notices when a change of the rule moves its shapes elsewhere.
#include "../gemm_impl.h"

// plan = {columns of a tile (256, 128, 64; 0: a weight-streaming kernel for few rows), workgroups that share a tile's K (slices
// of K there), 128-k macro steps of each but a shorter last one}.  `may_split`: the caller brings room for partial sums.
extern "C" int mase_bench_scaled_plan(int64_t M, int64_t N, int64_t K, int cus, int may_split, int* plan) {
    if (!plan || M < 1 || N < 1 || K < 512 || K % 256 != 0 || M > 0x7FFFFFFF || N > 0x7FFFFFFF || K >= ((int64_t)1 << 27) || cus < 8) return -1;
    const mase::ScaledMidPlan few = mase::plan_scaled_few((int)M, (int)N, (int)K, cus, may_split != 0);
    if (few.bn != 0) {
        plan[0] = few.bn;
        plan[1] = few.splits;
        plan[2] = few.mac_per;
        return 0;
    }
    const int slices = may_split ? mase::scaled_rows_slices((int)M, (int)N, (int)K) : 0;
    if (slices > 0 || mase::scaled_rows_shape_ok((int)M, (int)K)) {
        plan[0] = 0;
        plan[1] = std::max(slices, 1);
        plan[2] = (int)(K / 128 + plan[1] - 1) / plan[1];
        return 0;
    }
    const mase::ScaledMidPlan p = mase::plan_scaled((int)M, (int)N, (int)K, cus, may_split != 0);
    plan[0] = p.bn;
    plan[1] = p.splits;
    plan[2] = p.mac_per;
    return 0;
}

// does an extract down the rows go in tiles of 64 columns?
extern "C" int mase_bench_strided_column_tiles(int64_t columns, int64_t nkb, int element_bytes) {
    return mase::strided_column_tiles(columns, nkb, element_bytes) ? 1 : 0;
}

// does an extract of 16-bit elements down the rows go two columns to a lane?  (bf16 whose extents are multiples of 128 goes before that)
extern "C" int mase_bench_strided_pair_tiles(int64_t inner, int64_t columns, int64_t nkb, int bf16) {
    return mase::strided_pair_tiles(inner, columns, nkb, bf16 != 0) ? 1 : 0;
}

// does a product without bias go to the kernel for short contractions?
extern "C" int mase_bench_short_k(int64_t M, int64_t N, int64_t K, int64_t batches) {
    return mase::short_k_shape_ok((int)M, (int)N, (int)K, (int)batches) ? 1 : 0;
}

// do products that no kernel of whole macro steps takes go to the tiles of any shape?  (else to the 256 x 256 kernel)
extern "C" int mase_bench_any_shape(int64_t M, int64_t N, int64_t K, int64_t batches, int cus) {
    return mase::any_pays(mase::plan_any((int)M, (int)N, (int)K, (int)batches, cus, 1), (int)M, (int)N, (int)K, (int)batches, cus) ? 1 : 0;
}
