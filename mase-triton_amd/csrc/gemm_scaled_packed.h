// Products with a weight of 4- or 6-bit codes held at their own width: the matrix instruction reads E2M1, E2M3 and E3M2 as they are (W) beside E4M3
// bytes (A), so a product that is bound by reading W reads half or three quarters of the bytes.
//
// The packed weight is laid out as the instruction takes it.  For these formats lane 16 g + r of a wavefront holds the 32 codes of block g of
// row r of a 16-row x 128-k tile (measured with a one-wavefront probe: consecutive k, code i at bits BITS i of the lane's registers, the
// lane's own scale), so the tile's fragment is 64 x 16 bytes (4 bits), or 64 x 16 bytes and then 64 x 8 (6 bits), one load instruction
// each, and the tiles follow each other along k: [rows_pad / 16][K / 128][1024 or 1536 bytes].  A wavefront's load is 1 KB in a row and what it
// brings are operands: nothing passes through LDS.  The scales are those of the prepared operand ([K / 128][rows_pad] dwords).
//
// mxfp_gemm_packed_few_kernel: up to 16 rows of A, K <= 16384; A in registers as in gemm_scaled_few.h, W straight to registers two slices ahead.
// From 17 rows: the tiles of gemm_scaled_mid.h, fragments by DMA.  Products alone, bytes -> packed, another W on every call, us (N x K): E2M1 12 rows of
// 14336 x 4096 13.8 -> 9.0, 48 rows 15.4 -> 9.1, 200 rows 23.8 -> 16.3; 48 rows of 4096 x 14336 18.2 -> 12.2; E3M2 48 and 200 rows of 14336 x 4096 15.3 ->
// 11.2 and 23.9 -> 17.5, 48 rows of 4096 x 14336 18.1 -> 14.6.  (E4M3 bytes in this order: level with rows of bytes, so it is not the order but the
// size.  Longer rings than the tiles of bytes have: 0.5 us slower.)  What bounds it: the same path into the CUs, 30 MB of W in 9 us, 5 of them latencies.
// (included after gemm_impl.h)
#pragma once

namespace mase {

template <int WF>
struct PackedSlice {
    typename WFragment<WF>::T w[32 / SRG_WAVES];   // this wavefront's macro steps of a slice
    uint32_t sc[32 / SRG_WAVES];
};

constexpr int PF_RED = 16 * SRR_ROW, PF_SCB = PF_RED + 2 * SRG_WAVES * 1024, PF_LUT = PF_SCB + 16 * 128;     // LDS: A, partial sums of two units, A's scale bytes, code table
constexpr int PF_LDS_BYTES = PF_LUT + 2048 + 16;
static_assert(PF_LDS_BYTES > 80 * 1024, "no CU is given two of these workgroups while another has none");

template <int SL, int XMODE, class XF, int WF>
__global__ __launch_bounds__(SF_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void mxfp_gemm_packed_few_kernel(
    const void* __restrict__ a, const uint32_t* __restrict__ a_scales, const uint8_t* __restrict__ w_codes, const uint32_t* __restrict__ w_scales,
    const void* __restrict__ bias, int bias_dtype, void* __restrict__ y, int M, int N, int K, int rows_a, int rows_w, int slice_macs,
    int full_rounds, int tail_halves) {
    constexpr int SPW = 32 / SRG_WAVES, W_FRAG = w_frag_bytes<WF>();
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    uint8_t* const tile = lds;
    uint8_t* const scb = lds + PF_SCB;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    const int nmac = K / 128, groups = (N + 15) / 16;
    const int units = rows_unit_count((int)blockIdx.x, (int)gridDim.x, groups, full_rounds, tail_halves);
    auto macs_of = [&](int j) __attribute__((always_inline)) { return min(slice_macs, nmac - j * slice_macs); };        // at least one (the launcher checks)

    // slice j of unit u; plain arithmetic instead of branches, as in gemm_scaled_few.h: lanes of rows that a half unit leaves out, and all lanes
    // past the last unit, read the first lane's line
    auto issue = [&](PackedSlice<WF>& c, int u, int j) __attribute__((always_inline)) {
        const RowsUnit ru = rows_unit((int)blockIdx.x, u, (int)gridDim.x, full_rounds, tail_halves);
        const uint32_t in = u < units ? 1u : 0u, mine = ru.half < 0 || (r >> 3) == ru.half ? in : 0u;
        const uint32_t group = in * (uint32_t)ru.group;
        const uint32_t lo = mine * 16u * lane, hi = 1024u + mine * 8u * lane;
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const uint8_t* const p = w_codes + ((size_t)group * nmac + in * (uint32_t)(j * slice_macs + min(SPW * wave + s, macs_of(j) - 1))) * W_FRAG;
            if constexpr (WF == W_E2M1) c.w[s] = __builtin_nontemporal_load(reinterpret_cast<const intx4*>(p + lo));
            else {
                typedef int intx2 __attribute__((ext_vector_type(2)));
                const intx4 v = __builtin_nontemporal_load(reinterpret_cast<const intx4*>(p + lo));
                const intx2 t = __builtin_nontemporal_load(reinterpret_cast<const intx2*>(p + hi));
                c.w[s] = intx6{v[0], v[1], v[2], v[3], t[0], t[1]};
            }
        }
#pragma unroll
        for (int s = 0; s < SPW; ++s)
            c.sc[s] = __builtin_nontemporal_load(w_scales + (size_t)(j * slice_macs + min(SPW * wave + s, macs_of(j) - 1)) * rows_w + group * 16 + r);
    };

    // ---- A: fragments and scale bytes of this wavefront's macro steps, once, as in gemm_scaled_few.h
    const uint8_t* const frag = tile + r * SRR_ROW + 16 * g;
    intx8 af[SL][SPW];
    uint32_t a_sc[SL][SPW], keep[SL][SPW];
#pragma unroll
    for (int j = 0; j < SL; ++j)
#pragma unroll
        for (int s = 0; s < SPW; ++s) keep[j][s] = SPW * wave + s < macs_of(j) ? 0xFFu : 0u;
    auto take_fragments = [&](int j) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < SPW; ++s) {
            const int ms = min(SPW * wave + s, macs_of(j) - 1);
            const intx4 lo = *reinterpret_cast<const intx4*>(frag + ms * 128), hi = *reinterpret_cast<const intx4*>(frag + ms * 128 + 64);
            af[j][s] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            if constexpr (XMODE != FEW_OPERAND) a_sc[j][s] = scb[r * 128 + ms * 4 + g];
        }
    };
    PackedSlice<WF> c0, c1;
    auto issue_first = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        issue(c0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        issue(c1, SL > 1 ? 0 : 1, SL > 1 ? 1 : 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (XMODE == FEW_OPERAND) {
        constexpr int RPW = 16 / SRG_WAVES;
        const uint8_t* const a_codes = static_cast<const uint8_t*>(a);
        intx4 areg[2][RPW][4];
        auto load_a = [&](int j) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < RPW; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    areg[j & 1][i][q] = *reinterpret_cast<const intx4*>(a_codes + (size_t)(RPW * wave + i) * K + (size_t)j * slice_macs * 128 +
                                                                        min(1024u * q + 16u * lane, (uint32_t)macs_of(j) * 128u - 16u));
#pragma unroll
            for (int s = 0; s < SPW; ++s) a_sc[j][s] = a_scales[(size_t)(j * slice_macs + min(SPW * wave + s, macs_of(j) - 1)) * rows_a + r];
        };
        load_a(0);
#pragma unroll
        for (int j = 0; j < SL; ++j) {
            __builtin_amdgcn_sched_barrier(0);
            if (j + 1 < SL) load_a(j + 1);
            if (j == SL - 1) issue_first();
            __builtin_amdgcn_sched_barrier(0);
            if (j > 0) __syncthreads();
#pragma unroll
            for (int i = 0; i < RPW; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q) *reinterpret_cast<intx4*>(tile + (RPW * wave + i) * SRR_ROW + 1024 * q + 16 * lane) = areg[j & 1][i][q];
            __syncthreads();
            take_fragments(j);
#pragma unroll
            for (int s = 0; s < SPW; ++s) a_sc[j][s] >>= 8 * g;
        }
    } else {
        const uint16_t* const x = static_cast<const uint16_t*>(a);
        const XF f{};
        uint8_t* const lut = lds + PF_LUT;
        auto load_x = [&](int j, int i) __attribute__((always_inline)) {
            return *reinterpret_cast<const uint4*>(x + (size_t)i * K + (size_t)j * slice_macs * 128 + min(8u * tid, (uint32_t)macs_of(j) * 128u - 8u));
        };
        uint4 raw = load_x(0, 0);
        issue_first();
        if (XMODE == FEW_MINIFLOAT && tid == 0) lut[LdsLut<XF, false>::BYTES] = (uint8_t)((1u << (XF{}.E() + XF{}.M())) - 1u);
        LdsLut<XF, false>::fill(lut);
        const uint32_t lut_addr = (uint32_t)(uintptr_t)lut;
#pragma unroll
        for (int j = 0; j < SL; ++j) {
            if (j > 0) __syncthreads();
#pragma unroll 1
            for (int i = 0; i < M; ++i) {
                const uint4 now = raw;
                if (i + 1 < M) raw = load_x(j, i + 1);
                else if (j + 1 < SL) raw = load_x(j + 1, 0);
                uint32_t w0, w1, scale;
                scaled_operand_step<XF, XMODE == FEW_MINIFLOAT>(now, f, lut_addr, w0, w1, scale);
                if (8 * tid < macs_of(j) * 128) {
                    *reinterpret_cast<uint2*>(tile + i * SRR_ROW + 8 * tid) = make_uint2(w0, w1);
                    if ((tid & 3) == 0) scb[i * 128 + (tid >> 2)] = (uint8_t)scale;
                }
            }
            __syncthreads();
            take_fragments(j);
        }
    }
#pragma unroll
    for (int j = 0; j < SL; ++j)
#pragma unroll
        for (int s = 0; s < SPW; ++s) a_sc[j][s] &= keep[j][s];

    floatx4 acc;
    // multiply a slice, ask for the next but one into its place
    auto step = [&](PackedSlice<WF>& c, int u, auto j_c) __attribute__((always_inline)) {
        constexpr int j = decltype(j_c)::value;
#pragma unroll
        for (int s = 0; s < SPW; ++s) mfma_packed_after_valu<WF>(acc, c.w[s], af[j][s], (c.sc[s] >> (8 * g)) & keep[j][s], a_sc[j][s]);
        __builtin_amdgcn_sched_barrier(0);
        issue(c, u + (j + 2) / SL, (j + 2) % SL);
        __builtin_amdgcn_sched_barrier(0);
    };
    // the wavefronts' partial sums of unit u meet in LDS (two places in turn: one barrier a unit); a wavefront, another for every unit, adds them (lane
    // l holds n = 4 (l >> 4) + v, m = l & 15) and stores
    auto finish = [&](int u) __attribute__((always_inline)) {
        asm volatile("s_nop 15\n\ts_nop 15" : "+v"(acc) :: "memory");     // the matrix unit's last results have left its pipeline
        float* const red = reinterpret_cast<float*>(lds + PF_RED) + (u & 1) * SRG_WAVES * 256;
        *reinterpret_cast<floatx4*>(red + wave * 256 + lane * 4) = acc;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();                                     // (loads from global memory stay in flight)
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        if (wave == (u & (SRG_WAVES - 1))) {
            const RowsUnit ru = rows_unit((int)blockIdx.x, u, (int)gridDim.x, full_rounds, tail_halves);
            floatx4 s = *reinterpret_cast<const floatx4*>(red + lane * 4);
#pragma unroll
            for (int w = 1; w < SRG_WAVES; ++w) s += *reinterpret_cast<const floatx4*>(red + w * 256 + lane * 4);
            const int n = ru.group * 16 + 4 * g, m = r;
            if (u < units && m < M && n < N && (ru.half < 0 || (g >> 1) == ru.half)) {
                float out[4] = {s[0], s[1], s[2], s[3]};
                const int valid = min(4, N - n);
                if (bias)
                    for (int v = 0; v < valid; ++v) out[v] += load_bias(bias, bias_dtype, n + v);
                store_out4<BF16>(y, (int64_t)m * N + n, out, true, valid);
            }
        }
    };
    const floatx4 zero = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    int u = 0;
    do {      // (at least one unit, and the compiler is to know: it moves the loads of the first behind a test for none, and so behind A's)
        acc = zero;
        if constexpr (SL == 1) {
            step(c0, u, IntC<0>{});
            finish(u);
            acc = zero;                              // (a unit past the end is gone through, so that the loads in flight can be counted)
            step(c1, ++u, IntC<0>{});
        } else {
            static_assert(SL % 2 == 0, "the two places of a slice alternate over a unit");
            static_for<SL / 2>([&](auto p_c) __attribute__((always_inline)) {
                constexpr int p = 2 * decltype(p_c)::value;
                step(c0, u, IntC<p>{});
                step(c1, u, IntC<p + 1>{});
            });
        }
        finish(u);
    } while (++u < units);
}

template <int XMODE, class XF, int WF>
int launch_gemm_packed_few(const void* a, const uint32_t* a_scales, const uint8_t* w_codes, const uint32_t* w_scales, const void* bias, int bias_dtype,
                           void* y, int M, int N, int K, hipStream_t s) {
    const int cus = device_cu_count();
    if (cus <= 0) return fail(ERR_RUNTIME, "cannot read the compute-unit count of the current device");
    const RowsDeal d = deal_row_groups((N + 15) / 16, cus);
    auto go = [&](auto sl) {
        constexpr int SL = decltype(sl)::value;
        auto kern = mxfp_gemm_packed_few_kernel<SL, XMODE, XF, WF>;
        static std::atomic<uint64_t> allowed{0};
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), PF_LDS_BYTES, allowed)) return rc;
        hipLaunchKernelGGL(kern, dim3((unsigned)d.grid), dim3(SF_THREADS), PF_LDS_BYTES, s, a, a_scales, w_codes, w_scales, bias, bias_dtype, y, M, N, K,
                           (M + 255) / 256 * 256, (N + 255) / 256 * 256, (K / 128 + SL - 1) / SL, d.full_rounds, d.tail_halves);
        return check_launch("mxfp_linear_packed");
    };
    return K <= 4096 ? go(IntC<1>{}) : K <= 8192 ? go(IntC<2>{}) : go(IntC<4>{});
}

// ---- which kernel, and whether the packed weight is the better form at all
inline bool packed_few_ok(int M, int N, int K, int cus) { return M <= 16 && K <= SF_MAX_K && (K >= 1280 || (N + 15) / 16 <= cus); }

// Tile and split of K from 17 rows on (and for a short K against many columns): prices in us, as in plan_scaled, fitted to all tiles and splits of 17000
// shapes (1 - 1600 rows, N and K of the layers and random ones, another W on every call): a step takes `step` with few CUs busy and `busy` more with
// all, a round `round` beside its steps.  The pick is 0.5 % from the best of them in the mean, 4 % at the 95th percentile.
struct PackedPrice { double step, busy, round, launch, split, per_split, sums; };
inline double packed_price(bool six, int M, int N, int K, int cus, int bm, int bn, int splits) {
    static constexpr PackedPrice prices[2][3] = {
        {{0.112, 0.054, 1.6, 2.6, 2.2, 1.5, -2.9}, {0.194, 0.039, 2.2, 2.25, 1.95, 0.85, -0.9}, {0.252, 0.067, 3.2, 2.55, 2.4, 0.53, -0.43}},
        {{0.138, 0.090, 1.75, 2.75, 2.2, 1.5, -2.9}, {0.227, 0.045, 2.45, 2.35, 1.95, 0.85, -0.9}, {0.270, 0.111, 2.25, 3.0, 2.4, 0.53, -0.43}}};
    const PackedPrice& p = prices[six][bm == 64 ? 0 : bn == 64 ? 1 : 2];
    const int per = (K / SMAC + splits - 1) / splits;
    const int64_t wgs = (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn) * splits;
    const double busy = std::min(1.0, (double)wgs / cus), sums_mb = (double)M * N * 4.0 / 1e6;
    return (double)((wgs + cus - 1) / cus) * (per * (p.step + p.busy * busy) + p.round) + p.launch +
           (splits > 1 ? p.split + std::max(0.0, p.per_split * splits + p.sums) * sums_mb : 0.0);
}
inline ScaledMidPlan plan_packed(bool six, int M, int N, int K, int cus, bool may_split, double* price = nullptr) {
    const int nmac = K / SMAC;
    ScaledMidPlan best{0, 0, 1, nmac};
    double best_t = 1e30;
    for (int t = 0; t < 3; ++t) {
        const int bm = t == 0 ? 64 : 128, bn = t == 2 ? 128 : 64;
        if ((bm == 64) != (M <= 64)) continue;
        const int64_t tiles = (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
        for (int want = 1; want <= 16; ++want) {
            const int per = (nmac + want - 1) / want;
            if (want > 1 && (!may_split || tiles * want > cus || per < 4)) break;
            if ((nmac + per - 1) / per != want) continue;
            const double cost = packed_price(six, M, N, K, cus, bm, bn, want);
            if (cost < best_t) { best_t = cost; best = ScaledMidPlan{bm, bn, want, per}; }
        }
    }
    if (price) *price = best_t;
    return best;
}
// the price of 256 x 256 tiles of bytes, which many rows are better on
inline double price_256(int M, int N, int K, int cus) {
    double best = 1e30;
    for (int want = 1; want <= 16; ++want)
        if (scaled_256_shares_ok(M, N, K / SMAC, want, cus)) best = std::min(best, scaled_256_price(M, N, K / SMAC, want, cus));
    return best;
}
// Is the packed weight faster than bytes for such a product?  A small weight is launches and latencies either way, and the 6-bit fragments are two loads
// and a half where bytes are two.  GEMM times, packed / bytes, geometric mean over shapes by N * K from 2^23, 2^24, 2^25: E2M1 up to 16 rows 0.88,
// 0.81, 0.70, 33 - 64 rows 0.86, 0.78, 0.63, 129 - 256 rows 0.86, 0.78, 0.73; 6 bits 1.03, 0.99, 0.86 up to 16 rows, 0.92, 0.90, 0.77 at 33 - 64, 0.89, 0.86,
// 0.81 at 129 - 256.  Of 10000 shapes that this rule sends here 1 % come out more than 2 % slower (worst 1.12).
// (Those are with W from memory.  With W in the memory-side cache 4 bits stay ahead, but 6 bits do not where the tiles of bytes are one round over up to
// 8192 k, bound by LDS: 65 - 256 rows of 4096 x 4096 10.5 / 11.0 us, 8192 x 2048 8.0 / 8.4, 14336 x 4096 17.6 / 17.6, but 28672 x 4096 at 160 rows 37 / 30
// and 4096 x 14336 22.4 / 20.1: bytes there.)
inline bool packed_pays(bool six, int M, int N, int K, int cus) {
    const int64_t codes = (int64_t)N * K;
    if (codes < (M <= 32 ? (six ? (int64_t)1 << 25 : (int64_t)1 << 23) : (six ? (int64_t)1 << 23 : (int64_t)1 << 22))) return false;
    if (six && M <= 16 && K > 8192 && K <= 12288) return false;      // (three slices of bytes against four of which one is mostly idle: 11.7 / 13.2 at 3240 x 10496)
    if (six && M > 64 && M <= 400 && K <= 8192 && (int64_t)((M + 127) / 128) * ((N + 127) / 128) <= cus) return false;
    if (M <= 256) return true;
    if (M > 1024) return false;
    double price;
    plan_packed(six, M, N, K, cus, true, &price);
    return price < 0.97 * price_256(M, N, K, cus);
}

// x quantised inside: a translation unit for each form of W
template <int WF>
int packed_few_x_unit(const void* x, int exp_bits, int frac_bits, int minifloat, const uint8_t* w_codes, const uint32_t* w_scales, const void* bias, int bias_dtype,
                      void* y, int M, int N, int K, hipStream_t s);

}  // namespace mase
