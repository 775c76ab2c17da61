// Block-scaled MXFP GEMM for tens to hundreds of rows of A (a large decode batch, a chunk of a prompt), operands in the prepared
// form of gemm_scaled.h, on tiles of 128 x 128 or 128 x 64; and of 64 x 64 for up to 64 rows (plan_scaled_few).
//
// At these sizes the 256 x 256 tiles of gemm_scaled.h leave most CUs without one (200 x 14336 outputs: 56 tiles for 256 CUs), and
// splitting K for more of them costs fp32 partial sums of 256-row tiles that are mostly padding.  Smaller tiles give every CU
// one; what they cost is operand traffic per flop: a 128 x 128 tile takes 32 KB L2 -> LDS and 64 KB LDS -> registers per 128 k for
// 512 cycles of MFMA.  Both are about what a CU's paths carry in that time, so the kernel is organised to keep them running:
//   * four wavefronts (2 x 2 of 64 x 64, or 4 x 1 of 32 x 64 when the tile is 64 columns wide), one workgroup per CU;
//   * codes and scale dwords global -> LDS by DMA into a ring of four stages (64 x 64: eight) of one 128-k macro step each, as many steps ahead;
//   * the fragments of macro step s + 1 are read from LDS into the other of two register sets while step s is multiplied: at
//     the one barrier per step every wavefront has its operands in registers, and the slot of step s is free for the step a ring ahead;
//   * every MFMA is followed by its share of the step's LDS reads and DMAs and a scheduling barrier, as in gemm_scaled.h.
// What bounds it: a macro step takes 0.61 us (128 columns; 0.43 with 64), of which MFMAs and LDS are 0.29 (0.18).  The rest is the
// vector-memory path.  A CU takes in 55 bytes per ns when some of them come from HBM, however deep the ring is (six stages:
// the same) and whichever wavefronts ask (A and W asked for by different ones: the same): what is in flight is returned in
// order, and A's L2 hits queue behind W's misses.  With W in L2 as well the step is at its LDS and MFMA time.  With every CU
// at work HBM's share per CU is the nearer limit (128 x 14336 x 4096: 59 MB of W in 19 us, launch included).
// N x K = 14336 x 4096: 19.2 / 24.6 / 24.8 us at 128 / 200 / 256 rows, against 28.5 / 35.4 / 43.7 on 256 x 256 tiles; 4096 x 4096: 14 /
// 16 / 16.5 / 23 at 128 / 256 / 512 / 1024 rows against 21 / 24 / 27 / 42; 4096 x 14336: 22 / 29 at 128 / 256 against 33 / 36.
// LDS rows are 128 bytes, the 16-byte piece c of row r at position c ^ ((r >> 1) & 7).
// (included from gemm_impl.h's namespace, after gemm_scaled.h's typedefs)

// How W's codes lie: bytes of the prepared operand, or packed (gemm_scaled_packed.h): the fragments of 16 rows x 128 k one after the other,
// 4 or 6 bits a code.
enum { W_BYTES8 = 0, W_E2M1 = 1, W_E2M3 = 2, W_E3M2 = 3 };
template <int WF> constexpr int w_frag_bytes() { return WF == W_BYTES8 ? 2048 : WF == W_E2M1 ? 1024 : 1536; }    // of 16 rows x 128 k

// bytes of one ring stage, stages of the ring (as many as LDS holds, an even number of at most eight), bytes of LDS
template <int BM, int BN, int WF = W_BYTES8> constexpr int smd_stage_bytes() { return BM * 128 + BN / 16 * w_frag_bytes<WF>() + 1024; }
template <int BM, int BN, int WF = W_BYTES8> constexpr int smd_ring() { return BM == 128 ? (WF == W_E2M1 || (WF != W_BYTES8 && BN == 64) ? 6 : 4) : 8; }
template <int BM, int BN, int WF = W_BYTES8> constexpr int smd_lds_bytes() { return smd_ring<BM, BN, WF>() * smd_stage_bytes<BM, BN, WF>(); }

typedef int intx6 __attribute__((ext_vector_type(6)));
template <int WF> struct WFragment { typedef intx8 T; };
template <> struct WFragment<W_E2M1> { typedef intx4 T; };
template <> struct WFragment<W_E2M3> { typedef intx6 T; };
template <> struct WFragment<W_E3M2> { typedef intx6 T; };

#define MASE_MFMA_W(PRE, POST) asm volatile(PRE "v_mfma_scale_f32_16x16x128_f8f6f4 %0, %1, %2, %0, %3, %4 op_sel_hi:[0,0,0]" POST : "+v"(c) : "v"(w), "v"(a), "v"(sw), "v"(sa))
template <int WF>
__device__ inline void mfma_scaled_v(floatx4& c, const typename WFragment<WF>::T& w, const intx8& a, uint32_t sw, uint32_t sa) {
    if constexpr (WF == W_BYTES8) MASE_MFMA_W("", "");
    else if constexpr (WF == W_E2M1) MASE_MFMA_W("", " cbsz:4");
    else if constexpr (WF == W_E2M3) MASE_MFMA_W("", " cbsz:2");
    else MASE_MFMA_W("", " cbsz:3");
}
// the same behind VALU writes of the scales (mfma_scaled_after_valu)
template <int WF>
__device__ inline void mfma_packed_after_valu(floatx4& c, const typename WFragment<WF>::T& w, const intx8& a, uint32_t sw, uint32_t sa) {
    if constexpr (WF == W_E2M1) MASE_MFMA_W("s_nop 3\n\t", " cbsz:4");
    else if constexpr (WF == W_E2M3) MASE_MFMA_W("s_nop 3\n\t", " cbsz:2");
    else MASE_MFMA_W("s_nop 3\n\t", " cbsz:3");
}
#undef MASE_MFMA_W
// for the lanes in `mask`: 16 bytes from (sbase + voff) to LDS lds_addr + 16 * lane (masked here and not by a branch: the LDS address has to
// stay in a scalar register)
__device__ inline void dma_16b_masked(uint32_t lds_addr, uint32_t voff, const void* sbase, uint64_t mask) {
    uint64_t saved;
    asm volatile("s_mov_b64 %0, exec\n\ts_mov_b64 exec, %4\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b64 exec, %0"
                 : "=&s"(saved) : "s"(lds_addr), "v"(voff), "s"(sbase), "s"(mask) : "memory");
}
// 256 bytes: 4 per lane from (sbase + voff) to LDS lds_addr + 4 * lane
__device__ inline void dma_64_dwords(uint32_t lds_addr, uint32_t voff, const void* sbase) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_addr), "v"(voff), "s"(sbase) : "memory");
}

template <int DT_OUT, int BM, int BN, int WF>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void mxfp_gemm_scaled_mid_kernel(
    const uint8_t* __restrict__ a_codes, const uint32_t* __restrict__ a_scales, const uint8_t* __restrict__ w_codes,
    const uint32_t* __restrict__ w_scales, const void* __restrict__ bias, int bias_dtype, void* __restrict__ y_all, int M, int N, int K,
    int rows_a, int rows_w, int tiles_m, int splits, int mac_per, int n_walks, int64_t y_split_bytes) {
    constexpr int WN = BN / 64, WM = 4 / WN, MI = BM / 16 / WM, NJ = 4;       // wavefronts along n and m; 16-row and 16-column tiles of one
    constexpr int W_FRAG = w_frag_bytes<WF>(), W_GROUPS = BN / 64;           // W packed: a wavefront brings the fragments of so many 16-row groups
    constexpr bool W_SIX = W_FRAG == 1536;                                   // ... of 6 bits: 16 bytes of each lane, then 8 of each
    constexpr int A_BYTES = BM * 128, W_BYTES = BN / 16 * W_FRAG, STAGE = smd_stage_bytes<BM, BN, WF>(), SC = A_BYTES + W_BYTES;
    constexpr int RING = smd_ring<BM, BN, WF>();
    constexpr int A_DMAS = A_BYTES / 4096, W_DMAS = WF == W_BYTES8 ? W_BYTES / 4096 : W_GROUPS + (W_SIX ? 1 : 0), OPS = A_DMAS + W_DMAS + 1;   // DMAs per wavefront and step: A, W, scales
    constexpr int W_READS = WF == W_E2M1 ? 1 : 2;                            // LDS reads of a W fragment
    constexpr int READS = W_READS * NJ + 2 * MI + MI + NJ, MFMAS = MI * NJ;
    constexpr int W_STEP = WF == W_BYTES8 ? 128 : W_FRAG;                    // bytes from one macro step to the next
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave / WN, wave_n = wave % WN;
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;

    // walk (tile, split of K): m-tile fastest, then the split.  Workgroups are dealt to the 8 XCDs in turn; XCD x takes the x-th
    // eighth of the walks, so those that share rows of W share an L2.
    const int walk = (int)((blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3));     // (the grid is a multiple of 8)
    if (walk >= n_walks) return;
    const int tile_m = walk % tiles_m, rest = walk / tiles_m;
    const int z = rest % splits, tile_n = rest / splits, m0 = tile_m * BM, n0 = tile_n * BN;
    const int mac0 = z * mac_per, nm = min(mac_per, K / 128 - mac0);   // this walk's macro steps (at least one)
    uint8_t* const y = static_cast<uint8_t*>(y_all) + (size_t)z * (size_t)y_split_bytes;

    // ---- DMA.  Data: lane l fills position l & 7 of row 8 d + (l >> 3) of the wavefront's rows, which must hold the row's piece
    //      (l & 7) ^ (row >> 1 & 7).  Wavefront w: rows BM / 4 w .. of A, BN / 4 w .. of W, and 64 of the scale dwords (A's, then W's).
    uint32_t voff[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
        voff[d] = (uint32_t)(8 * d + (lane >> 3)) * (uint32_t)K + (uint32_t)(((lane & 7) ^ ((4 * d + (lane >> 4)) & 7)) << 4);
    const uint32_t sc_voff = (uint32_t)lane * 4u;
    const int sc_wave = min(wave, BM / 64 + BN / 64 - 1);               // (fewer than 256 dwords: the last wavefronts repeat W's)
    constexpr int SC_A = BM / 64;
    const uint8_t* pa = a_codes + (size_t)(m0 + BM / 4 * wave) * K + (size_t)mac0 * 128;
    const uint8_t* pw = WF == W_BYTES8 ? w_codes + (size_t)(n0 + BN / 4 * wave) * K + (size_t)mac0 * 128
                                       : w_codes + ((size_t)(n0 / 16 + W_GROUPS * wave) * (K / 128) + mac0) * W_FRAG;
    uint32_t w_voff[W_DMAS];                                           // packed: the groups' fragments, each as it lies
    if constexpr (WF != W_BYTES8) {
        const uint32_t group = (uint32_t)(K / 128) * W_FRAG;
#pragma unroll
        for (int d = 0; d < W_GROUPS; ++d) w_voff[d] = d * group + 16u * lane;
        if constexpr (W_SIX) w_voff[W_GROUPS] = (W_GROUPS == 2 ? (uint32_t)(lane >> 5) * group : 0u) + 1024u + 16u * (lane & 31);
    }
    const uint32_t* psc = sc_wave < SC_A ? a_scales + (size_t)mac0 * rows_a + m0 + 64 * sc_wave : w_scales + (size_t)mac0 * rows_w + n0 + 64 * (sc_wave - SC_A);
    const int sc_step = sc_wave < SC_A ? rows_a : rows_w;
    // workgroups of different columns start at different macro steps and wrap around: rows of W (and of A) are K bytes apart, and at
    // one k all of them would sit on the same few channels of the L2
    int at = tile_n % nm;                                             // the macro step that is issued next
    pa += (size_t)at * 128;
    pw += (size_t)at * W_STEP;
    psc += (size_t)at * sc_step;
    auto dma = [&](auto slot_c, auto q_c) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_c)::value, q = decltype(q_c)::value;
        if constexpr (q < A_DMAS) dma_1kb(lds_base + (uint32_t)(slot * STAGE + q * 1024) + (uint32_t)wave * (A_DMAS * 1024u), voff[q], pa);
        else if constexpr (q < A_DMAS + W_DMAS && WF == W_BYTES8) dma_1kb(lds_base + (uint32_t)(slot * STAGE + A_BYTES + (q - A_DMAS) * 1024) + (uint32_t)wave * (W_DMAS * 1024u), voff[q - A_DMAS], pw);
        else if constexpr (q < A_DMAS + W_GROUPS) dma_1kb(lds_base + (uint32_t)(slot * STAGE + A_BYTES + (q - A_DMAS) * 1024) + (uint32_t)wave * (W_GROUPS * 1024u), w_voff[q - A_DMAS], pw);
        else if constexpr (q < A_DMAS + W_DMAS) {
            const uint32_t to = lds_base + (uint32_t)(slot * STAGE + A_BYTES + BN * 64) + (uint32_t)wave * (W_GROUPS * 512u);
            if constexpr (W_GROUPS == 2) dma_1kb(to, w_voff[q - A_DMAS], pw);
            else dma_16b_masked(to, w_voff[q - A_DMAS], pw, 0x00000000FFFFFFFFull);
        }
        else dma_64_dwords(lds_base + (uint32_t)(slot * STAGE + SC) + (uint32_t)sc_wave * 256u, sc_voff, psc);
    };
    auto advance = [&]() __attribute__((always_inline)) {
        const bool wrap = ++at == nm;
        at = wrap ? 0 : at;
        pa += wrap ? -(int64_t)(nm - 1) * 128 : 128;
        pw += wrap ? -(int64_t)(nm - 1) * W_STEP : W_STEP;
        psc += wrap ? -(int64_t)(nm - 1) * sc_step : sc_step;
    };

    // ---- fragments: lane (g = l >> 4, r = l & 15) reads pieces g and g + 4 of row r of its 16-row tile, and the row's scale byte g
    const uint32_t f_off = (uint32_t)(lane & 15) * 128u + (uint32_t)((((lane >> 4) ^ ((lane >> 1) & 7)) & 7) << 4);
    const uint8_t* const a_lo = lds + wave_m * (MI * 2048) + f_off;
    const uint8_t* const a_hi = lds + wave_m * (MI * 2048) + (f_off ^ 64u);
    // (packed: the lane's 32 codes, block g of row r, as they lie)
    const uint8_t* const w_lo = lds + A_BYTES + (WF == W_BYTES8 ? wave_n * (NJ * 2048) + f_off : wave_n * (NJ * 1024) + 16u * lane);
    const uint8_t* const w_hi = lds + A_BYTES + wave_n * (NJ * 2048) + (f_off ^ 64u);        // (bytes)
    constexpr int W_LO = WF == W_BYTES8 ? 2048 : 1024;               // from one fragment to the next
    // (6 bits: the second parts' places, hidden from the compiler: it would read two of them with one instruction and copy them apart)
    uint32_t w_hi6[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        w_hi6[j] = (uint32_t)(A_BYTES + BN * 64 + (wave_n * NJ + j) * 512 + 8 * lane);
        if (W_SIX) asm volatile("" : "+v"(w_hi6[j]));
    }
    const uint8_t* const a_sc = lds + SC + wave_m * (MI * 64) + (lane & 15) * 4 + (lane >> 4);
    const uint8_t* const w_sc = lds + SC + BM * 4 + wave_n * (NJ * 64) + (lane & 15) * 4 + (lane >> 4);
    floatx4 acc[NJ][MI];
    intx8 af[2][MI];
    typename WFragment<WF>::T wf[2][NJ];
    uint32_t as[2][MI], ws[2][NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i) acc[j][i] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // read k (0 .. READS - 1) of the stage in `slot` into register set `set`: W fragment 0, A fragment 0, W 1, A 1, ..., then scales
    auto read = [&](auto slot_c, auto set_c, auto k_c) __attribute__((always_inline)) {
        constexpr int slot = decltype(slot_c)::value, set = decltype(set_c)::value, k = decltype(k_c)::value;
        constexpr int W_ALL = W_READS * NJ;
        if constexpr (k < W_ALL) {
            constexpr int j = k / W_READS;
            const uint8_t* const from_lo = w_lo + slot * STAGE + j * W_LO;
            if constexpr (WF == W_E2M1) wf[set][j] = *reinterpret_cast<const intx4*>(from_lo);
            else if constexpr (W_SIX) {
                if constexpr (k % 2 == 0) {
                    const intx4 v = *reinterpret_cast<const intx4*>(from_lo);
                    wf[set][j] = __builtin_shufflevector(v, v, 0, 1, 2, 3, -1, -1);
                } else {
                    const int2 v = *reinterpret_cast<const int2*>(lds + w_hi6[j] + slot * STAGE);
                    wf[set][j][4] = v.x;
                    wf[set][j][5] = v.y;
                }
            } else if constexpr (k % 2 == 0) wf[set][j].lo = *reinterpret_cast<const intx4*>(from_lo);
            else wf[set][j].hi = *reinterpret_cast<const intx4*>(w_hi + slot * STAGE + j * W_LO);
        } else if constexpr (k < W_ALL + 2 * MI) {
            constexpr int i = (k - W_ALL) / 2;
            if constexpr ((k - W_ALL) % 2 == 0) af[set][i].lo = *reinterpret_cast<const intx4*>(a_lo + slot * STAGE + i * 2048);
            else af[set][i].hi = *reinterpret_cast<const intx4*>(a_hi + slot * STAGE + i * 2048);
        } else if constexpr (k < W_ALL + 2 * MI + NJ) {
            constexpr int j = k - W_ALL - 2 * MI;
            ws[set][j] = w_sc[slot * STAGE + j * 64];
        } else {
            constexpr int i = k - W_ALL - 2 * MI - NJ;
            as[set][i] = a_sc[slot * STAGE + i * 64];
        }
    };

    static_for<RING>([&](auto s_c) __attribute__((always_inline)) {
        static_for<OPS>([&](auto q_c) __attribute__((always_inline)) { dma(s_c, q_c); });
        advance();
    });
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 1) * OPS) : "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    static_for<READS>([&](auto k_c) __attribute__((always_inline)) { read(IntC<0>{}, IntC<0>{}, k_c); });

    for (int base = 0; base < nm; base += RING) {
        static_for<RING>([&](auto u_c) __attribute__((always_inline)) {
            constexpr int u = decltype(u_c)::value, set = u & 1, next = (u + 1) % RING;
            if (base + u < nm) {
                // stage s + 1 of this wavefront has landed (the RING - 2 stages behind it may still fly), step s is in registers
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"((RING - 2) * OPS) : "memory");
                lds_barrier();
                asm volatile("" ::: "memory");
                static_for<MFMAS>([&](auto t_c) __attribute__((always_inline)) {
                    constexpr int t = decltype(t_c)::value, i = t / NJ, j = t % NJ;
                    mfma_scaled_v<WF>(acc[j][i], wf[set][j], af[set][i], ws[set][j], as[set][i]);
                    constexpr int r0 = t * READS / MFMAS, r1 = (t + 1) * READS / MFMAS, d0 = t * OPS / MFMAS, d1 = (t + 1) * OPS / MFMAS;
                    static_for<r1 - r0>([&](auto k_c) __attribute__((always_inline)) { read(IntC<next>{}, IntC<set ^ 1>{}, IntC<r0 + decltype(k_c)::value>{}); });
                    static_for<d1 - d0>([&](auto k_c) __attribute__((always_inline)) { dma(IntC<u>{}, IntC<d0 + decltype(k_c)::value>{}); });
                    __builtin_amdgcn_sched_barrier(0);
                });
                advance();
            }
        });
    }
    // the look-ahead DMAs still target LDS, which the outputs pass through
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");      // the matrix unit's last results have left its pipeline
    lds_barrier();
    asm volatile("" ::: "memory");

    // ---- output: lane holds, for tile (j, i), y[m][n .. n+3] with m = 16 i + lane % 16, n = 16 j + 4 (lane / 16) of the wavefront's
    //      outputs; staged so that a store instruction writes whole lines (128 bytes of a row: 64 columns, 32 of fp32)
    constexpr int OB = DT_OUT == F32 ? 4 : 2, PASSES = DT_OUT == F32 ? 2 : 1, JT = NJ / PASSES;
    uint8_t* const out = lds + wave * (MI * 2048);
    const int g = lane >> 4, r = lane & 15;
    const int row0 = m0 + wave_m * (MI * 16), col0 = n0 + wave_n * 64;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
#pragma unroll
        for (int jj = 0; jj < JT; ++jj) {
            const int j = p * JT + jj;
            float b[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            if (bias) {
#pragma unroll
                for (int v = 0; v < 4; ++v) b[v] = load_bias(bias, bias_dtype, min(col0 + 16 * j + 4 * g + v, N - 1));
            }
#pragma unroll
            for (int i = 0; i < MI; ++i) {
                const floatx4 c = acc[j][i];
                uint8_t* const row = out + (16 * i + r) * 128;
                if constexpr (DT_OUT == F32)
                    *reinterpret_cast<float4*>(row + (((4 * jj + g) ^ (r & 7)) * 16)) = make_float4(c[0] + b[0], c[1] + b[1], c[2] + b[2], c[3] + b[3]);
                else
                    *reinterpret_cast<uint2*>(row + (((2 * jj + (g >> 1)) ^ (r & 7)) * 16) + (g & 1) * 8) = pack_out4<DT_OUT>(c[0] + b[0], c[1] + b[1], c[2] + b[2], c[3] + b[3]);
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the wavefront's own writes)
        const int col = col0 + p * 32 + (lane & 7) * (16 / OB);
#pragma unroll
        for (int t = 0; t < MI * 2; ++t) {
            const int row = 8 * t + (lane >> 3);
            const u32x4 v = *reinterpret_cast<const u32x4*>(out + row * 128 + (((lane & 7) ^ (row & 7)) * 16));
            if (row0 + row < M && col < N) *reinterpret_cast<u32x4*>(y + ((size_t)(row0 + row) * N + col) * OB) = v;
        }
        asm volatile("" ::: "memory");
    }
}

struct ScaledMidPlan {
    int bm;        // rows of a tile: 64, 128; 256: the 256 x 256 kernel of gemm_scaled.h
    int bn;        // columns of a tile: 128 or 64; 256: the 256 x 256 kernel of gemm_scaled.h
    int splits;    // workgroups that share a tile's K, each with its own fp32 [M, N] array of the workspace
    int mac_per;   // macro steps per split
};

// Which tile, and how many workgroups share its K.  Every candidate is priced, in us: rounds of workgroups over the CUs x macro
// steps x time of a step, plus launch, prologue and epilogue, plus, when K is split, the second launch and the partial sums
// written and read once.  Fitted to both kernels forced on N = 1024 .. 14336, K = 1024 .. 14336, 65 .. 2048 rows: a step takes 1.0 us
// (256 x 256) with few CUs busy and 1.2 with all, 0.62 (128 x 128) either way, 0.37 and 0.46 (128 x 64); the 256 x 256 kernel walks
// its tiles as one stream (8 us once), the others pay 2.5 us per round and 2 once.  Where prices are close so are the
// kernels: 384 x 14336 x 4096 takes 43.4 us on 256 x 256 tiles and 44.0 on 128 x 128 ones, 2048 x 4096 x 4096 41 and 45.
// Up to 1600 rows, 8192 columns and 4096 k the smaller tiles are priced by a later fit, another W on every call (3500 shapes of 65 - 1600 rows, 7 %): a step takes
// 0.22 us (128 x 64) and 0.29 (128 x 128) with few CUs busy, 0.32 and 0.49 with all.  It moves products of few columns from many shares of K
// to whole 128 x 64 tiles (150 x 4096 x 4096 13.7 -> 11.5 us, 700 x 1024 x 4096 13.8 -> 10.3).  They have to be a fifth below the 256 x 256 kernel, whose
// price errs the other way on a long K and on a W in the memory-side cache (671 x 4096 x 14336: 54.1 us in four shares, 58.6 on 128 x 128; a SwiGLU
// block of 680 x 4096 x 12288 155 / 163); of a longer K the gain over all shapes was 1 %.  Elsewhere the figures above.
// One row of the smaller tiles (up to 128 rows of A) shares nothing of W: a second round adds a wait, up to 1.4 us when it is full (128 x
// 65536, K = 512 / 1024 / 2048: 14.6 / 19.5 / 29.3 us on 128 x 128 tiles, 12.8 / 17.7 / 27.2 on one round of 256 x 256 ones, fp32 out 18.0 / 23.4 / 33.1
// and 14.3 / 19.5 / 28.6; K = 4096 53 and 55).
// the price of `splits` equal shares of K on 256 x 256 tiles
inline double scaled_256_price(int M, int N, int nmac, int splits, int cus) {
    const int64_t wgs = (int64_t)((M + SM - 1) / SM) * ((N + SN - 1) / SN) * splits;
    const double busy = wgs >= cus ? 1.0 : (double)wgs / cus, sums_mb = (double)M * N * 4.0 / 1e6;
    return (double)((wgs + cus - 1) / cus) * (nmac / splits * (1.0 + 0.2 * busy)) + 8.0 + (splits > 1 ? 3.0 + (2.0 * splits + 0.5) * sums_mb * 0.16 : 0.0);
}
inline bool scaled_256_shares_ok(int M, int N, int nmac, int splits, int cus) {      // (that kernel walks equal shares of pairs of macro steps)
    return splits == 1 || ((int64_t)((M + SM - 1) / SM) * ((N + SN - 1) / SN) * splits <= cus && nmac % splits == 0 && nmac / splits % 2 == 0 && nmac / splits >= 4);
}
inline ScaledMidPlan plan_scaled(int M, int N, int K, int cus, bool may_split) {
    const int nmac = K / SMAC;
    ScaledMidPlan best{256, 256, 1, nmac};
    if (cus <= 0) return best;
    const bool few_columns = M <= 1600 && N <= 8192 && K <= 4096;
    const double mn_mb = (double)M * N * 4.0 / 1e6;
    double best_t = 1e30;
    for (int want = 1; want <= (may_split ? 16 : 1); ++want) {
        if (!scaled_256_shares_ok(M, N, nmac, want, cus)) continue;
        if (const double t = scaled_256_price(M, N, nmac, want, cus); t < best_t) { best_t = t; best = ScaledMidPlan{256, 256, want, nmac / want}; }
    }
    for (int bn = 128; bn >= 64; bn /= 2) {
        const int64_t tiles = (int64_t)((M + 127) / 128) * ((N + bn - 1) / bn);
        for (int want = 1; want <= 16; ++want) {
            if (want > 1 && (!may_split || tiles * want > cus)) break;
            const int per = (nmac + want - 1) / want;
            if (want > 1 && (per < 4 || (nmac + per - 1) / per != want)) continue;
            const int64_t wgs = tiles * want;
            const double busy = wgs >= cus ? 1.0 : (double)wgs / cus;
            const double step = bn == 128 ? 0.62 : 0.37 + 0.09 * busy;
            const double rounds = (double)((wgs + cus - 1) / cus);
            const double unshared = M <= 128 && wgs > cus ? 1.4 * std::min(1.0, (double)(wgs - cus) / cus) : 0.0;
            double t = rounds * (per * step + 2.5) + (2.0 + unshared) + (want > 1 ? 3.0 + (2.0 * want + 0.5) * mn_mb * 0.16 : 0.0);
            if (bn == 128 && few_columns)
                t = 1.25 * (rounds * (per * (0.292 + 0.195 * busy) + 0.77) + 4.65 + unshared + (want > 1 ? 2.9 + std::max(0.0, 0.55 * want - 0.8) * mn_mb : 0.0));
            else if (bn == 64 && few_columns)
                t = 1.25 * (rounds * (per * (0.222 + 0.097 * busy) + 1.3) + 3.35 + unshared + (want > 1 ? 2.4 + std::max(0.0, 0.75 * want - 1.0) * mn_mb : 0.0));
            if (t < best_t) { best_t = t; best = ScaledMidPlan{128, bn, want, per}; }
        }
    }
    return best;
}

// Up to 64 rows: tiles of 64 x 64 against the weight-streaming kernel that keeps A in its registers.  The latter's prologue and the MFMAs
// of a unit grow with the 16-row tiles of A (every CU takes in all of A), and a unit of a short K is too few bytes in flight; these
// tiles read 64 rows of A per 64 of W whatever M is, from a grid of N / 64.  Prices in us with W from memory.  GEMMs alone, W from memory |
// W in the memory-side cache, tiles / the other kernel: 14336 x 4096 32 rows 16.7 / 16.0 | 12.9 / 15.4, 48 rows 16.8 / 17.5 | 13.0 / 17.0, 64 rows
// 16.9 / 19.5 | 13.0 / 19.3; 4096 x 14336, K in four, 32 rows 19.2 / 18.5 | 17.4 / 18.3, 48 rows 19.5 / 20.5 | 17.6 / 20.4, 64 rows 19.8 / 23.0 | 17.7 / 23.1;
// 8192 x 2048 16 rows 7.1 / 7.8 | 7.1 / 7.5, 64 rows 7.1 / 12.1 | 7.1 / 11.8; 4096 x 4096 32 rows 9.4 / 8.1 | 9.4 / 7.5, 64 rows 9.4 / 10.3 | 9.4 / 9.7.  Layer calls
// of 48 rows, before and now: 14336 x 768 18.2 / 8.7, 8192 x 8192 27.3 / 21.5, 2176 x 10752 18.1 / 15.6.  (Tiles of 64 x 128 are never ahead: 14336 x
// 4096 21.2 | 13.8.)  bn == 0: a weight-streaming kernel.
// The tiles' price for K up to 4096 is fitted to the operand of x and the product, another W on every call (where the tiles lose more than
// alone), by the other kernel's operand tiles: of 2100 shapes eight come out more than 2 % slower than on the other kernel (worst 49 x 4096 x
// 3072, 14.8 / 13.3), 145 with the price of a longer K for all.  Tiles / the other kernel, us: 17 x 8192 x 2560 14.6 / 12.3, 1 x 8192 x 2048
// 11.7 / 10.1, 32 x 32768 x 2560 29.2 / 25.2, 5 x 93008 x 1792 50.7 / 43.9, 64 x 65536 x 3072 58.4 / 52.4, but 16 x 14336 x 768 9.0 / 13.0, 17 x 65536 x 512
// 22 / 35, 64 x 14336 x 4096 20.6 / 23.9.
inline ScaledMidPlan plan_scaled_few(int M, int N, int K, int cus, bool may_split) {
    const int nmac = K / SMAC;
    ScaledMidPlan best{0, 0, 1, nmac};
    if (M > 64 || cus <= 0) return best;
    // 17 - 32 rows of a long K: level at best (896 x 14336 13.4 / 14.7); up to 16 rows gemm_scaled_few.h, with no room for sums the chunked kernel
    if (M <= 32 && K > 4096) return best;
    const double mn_mb = (double)M * N * 4.0 / 1e6;
    auto split_cost = [&](int splits) { return splits > 1 ? 3.0 + (2.0 * splits + 0.5) * mn_mb * 0.16 : 0.0; };
    // the other kernel: prologue, then units of 16 rows of W x (a slice of) K, the last as half units; a unit takes its latency at least
    const int slices = K > 4096 ? (may_split ? scaled_rows_slices(M, N, K) : 0) : 1;
    double best_t = 1e30;                                   // (33 rows and more without room for its sums: these tiles)
    if (slices > 0) {
        const int mt = (M + 15) / 16, groups = (N + 15) / 16, per_slice = std::max(1, std::min(groups, cus / slices));
        const double units = slices > 1 ? (groups + per_slice - 1) / per_slice : std::max(1.0, std::ceil(2.0 * groups / cus) / 2.0);
        const double busy = std::min(1.0, (double)groups * slices / cus);
        best_t = 3.8 + 0.9 * mt * (0.5 + 0.5 * busy) + units * (std::max(1.6, (double)nmac / slices / 32.0 * 2.15) * (0.4 + 0.6 * busy) + 0.25 * mt) +
                 split_cost(slices) - 0.5;
    }
    struct Price { double step, busy, round, launch; };
    const Price price = K > 4096  ? Price{0.15, 0.28, 1.2, 2.0}
                        : M <= 16 ? Price{0.24, 0.36, 1.2, 2.0}
                        : M <= 32 ? Price{0.21, 0.36, 1.2, 1.5}
                        : M <= 48 ? Price{0.15, 0.28, 2.1, 1.1}
                                  : Price{0.19, 0.32, 1.8, 0.5};
    const int64_t tiles = (N + 63) / 64;
    for (int want = 1; want <= 16; ++want) {
        if (want > 1 && (!may_split || tiles * want > cus || N % 4 != 0)) break;
        const int per = (nmac + want - 1) / want;
        if (want > 1 && (per < 12 || (nmac + per - 1) / per != want)) continue;
        const int64_t wgs = tiles * want;
        const double busy = wgs >= cus ? 1.0 : (double)wgs / cus;
        const double t = (double)((wgs + cus - 1) / cus) * (per * (price.step + price.busy * busy) + price.round) + price.launch + split_cost(want);
        if (t < best_t) { best_t = t; best = ScaledMidPlan{64, 64, want, per}; }
    }
    return best;
}

template <int DT_OUT, int WF = W_BYTES8>
int launch_gemm_scaled_mid(const uint8_t* a_codes, const uint32_t* a_scales, const uint8_t* w_codes, const uint32_t* w_scales, const void* bias,
                           int bias_dtype, void* y, int M, int N, int K, const ScaledMidPlan& p, void* workspace, hipStream_t s) {
    const int rows_a = (M + 255) / 256 * 256, rows_w = (N + 255) / 256 * 256;
    const int tiles_m = (M + p.bm - 1) / p.bm, tiles_n = (N + p.bn - 1) / p.bn;
    const int64_t walks = (int64_t)tiles_m * tiles_n * p.splits, mn = (int64_t)M * N;
    if (walks >= (1 << 30)) return fail(ERR_UNSUPPORTED, "too many tiles");
    auto go = [&](auto kern, int lds_bytes, std::atomic<uint64_t>& allowed, void* out, int64_t split_bytes, const void* b) {
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, allowed)) return rc;
        hipLaunchKernelGGL(kern, dim3((unsigned)((walks + 7) / 8 * 8)), dim3(256), lds_bytes, s, a_codes, a_scales, w_codes, w_scales, b, bias_dtype, out, M,
                           N, K, rows_a, rows_w, tiles_m, p.splits, p.mac_per, (int)walks, split_bytes);
        return check_launch("mxfp_gemm_scaled");
    };
    static std::atomic<uint64_t> allowed[2][2][2] = {};
    auto pick = [&](auto dt, void* out, int64_t split_bytes, const void* b) {
        constexpr int DT = decltype(dt)::value;
        std::atomic<uint64_t>* const done = allowed[split_bytes != 0][p.bm == 64];
        if (p.bm == 64) return go(mxfp_gemm_scaled_mid_kernel<DT, 64, 64, WF>, smd_lds_bytes<64, 64, WF>(), done[0], out, split_bytes, b);
        return p.bn == 128 ? go(mxfp_gemm_scaled_mid_kernel<DT, 128, 128, WF>, smd_lds_bytes<128, 128, WF>(), done[0], out, split_bytes, b)
                           : go(mxfp_gemm_scaled_mid_kernel<DT, 128, 64, WF>, smd_lds_bytes<128, 64, WF>(), done[1], out, split_bytes, b);
    };
    if (p.splits == 1) return pick(IntC<DT_OUT>{}, y, 0, bias);
    if (int rc = pick(IntC<F32>{}, workspace, mn * 4, nullptr)) return rc;
    hipLaunchKernelGGL(split_k_reduce_kernel<DT_OUT>, dim3((unsigned)((mn / 4 + 255) / 256)), dim3(256), 0, s, static_cast<const float*>(workspace), p.splits,
                       mn, N, bias, bias_dtype, y);
    return check_launch("mxfp_gemm_scaled");
}
