// MXFP GEMM kernel for gfx950 for a short contraction (K <= 128): dense bf16 A, MXFP W, one or many products per launch
// (attention scores are batch x heads products with K = the head dimension and thousands of outputs per row of W).
//
// With K <= 128 a tile is a handful of MFMAs and the time is the outputs' way to memory, so everything is built around that.
// A workgroup walks down m-tiles of 64 rows of A against 128 rows of W:
//   * W is composed once per column of tiles, straight into the registers that the MFMAs read (a lane loads the 8 codes per
//     16 k that it will feed), and stays there: no LDS, no barrier, no second compose for the next tile;
//   * a 64-row A tile comes global -> LDS by DMA into one of two stages, one tile ahead;
//   * four wavefronts, 2 (rows) x 2 (columns), 32 x 64 outputs each: 2 MFMAs (32x32x16) per 16 k from one A fragment;
//   * the outputs pass through a wave-private piece of LDS and leave as whole 128-byte runs of a row, 16 bytes per lane,
//     in buffer stores: rows past M and columns past N are dropped by the bounds check of the store, without a branch, so
//     the number of stores per tile is known and the wait for the next A tile does not wait for this tile's stores.
// Two workgroups per CU with equal runs of tiles cover each other's phases.  (Three, which LDS and registers would hold, get
// into each other's way in L2: 33 against 60 us at 1001 rows of the shape below, 56 against 67 at 2048 x 2048.)
// Any M and N, K a multiple of 32 (short_k_shape_ok in gemm_impl.h says which it is for).  64 products of 1000 x 1000 x 128 (E4M3, bf16
// out, 152 MB to read and write), repeated on the same buffers: 32 us, 4.7 TB/s (a plain copy of that many bytes reaches 5.2); with other
// operands and outputs on every call, as in a model, 52 us.  At 1024 x 1024 that is 28 and 30 us (992: 49, 1008: 51): rows of whole
// lines are stored past the caches, others fill these with y, and operands that have to come from memory wait behind its
// write-back (fresh outputs alone, the operands at hand: 33 us; what reaches memory is y in 64-byte requests in both cases).  32
// products of 2048 x 2048 x 128: 49 and 52 us, 5.6 TB/s.  The kernels that took such shapes before (the
// 128 x 128 x 32 single-buffer one, the 512 x 128 one with products as grid planes) take 98, 128 and 259 us on fresh buffers.
#pragma once
#include "gemm_impl.h"

namespace mase {

constexpr int SH_M = 64, SH_N = 128, SH_MAX_K = 128;
constexpr int SH_STAGE_OUT = 32 * 128;                    // bytes of a wavefront's output staging: 32 rows x 128 B

// KP: the K the loops are built for (64 or 128); a smaller K is filled up with zeros on both sides.
template <class FW, int DT_OUT, int KP>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void mxfp_gemm_short_k_kernel(
    const uint16_t* __restrict__ a_dense, const uint8_t* __restrict__ w_scales, const uint8_t* __restrict__ w_elements, void* __restrict__ y_all,
    int M, int N, int K, int n_tiles, int m_tiles, uint32_t per_run, uint32_t longer_runs, GemmBatch gb) {
    constexpr int Q = KP / 16;                             // 16-k steps
    constexpr int ROW = 2 * KP;                            // bytes of an A row in LDS
    constexpr int STAGE = SH_M * ROW;                      // one A tile
    constexpr int DMAS = STAGE / 1024 / 4;                 // per wavefront and tile
    constexpr int ROWS_PER_DMA = 1024 / ROW, CHUNKS = ROW / 16;
    constexpr int ESZ = DT_OUT == F32 ? 4 : 2, PASSES = DT_OUT == F32 ? 2 : 1, STORES = 4 * PASSES;   // 16-byte stores per lane and tile
    __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * STAGE + 4 * SH_STAGE_OUT];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave >> 1, wave_n = wave & 1, g2 = lane >> 5, r32 = lane & 31;
    // The tiles (product, n-tile, m-tile; m fastest) are dealt to the workgroups in equal contiguous runs, so that no CU is
    // left with a last round of its own.  Workgroups are dealt to the 8 XCDs in turn; XCD x takes the x-th eighth of the runs:
    // the workgroups that read the same A tiles share an L2.
    const uint32_t run = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);   // (the grid is a multiple of 8)
    const uint32_t t0 = run * per_run + min(run, longer_runs), t1 = t0 + per_run + (run < longer_runs ? 1u : 0u);
    if (t0 >= t1) return;
    const uint32_t lds_addr = (uint32_t)(uintptr_t)lds;

    // A DMA: an instruction moves 1 KB; lane l fills position l % CHUNKS of row l / CHUNKS (of the instruction's rows), which
    // must hold chunk position ^ swizzle(row): conflict-free 128-bit fragment reads.  Rows past M re-read row M - 1.
    auto swizzle = [](int row) { return KP == 128 ? (row & 15) : ((row >> 1) & 7); };
    int a_row[DMAS];
    uint32_t a_chunk[DMAS];
    bool a_live[DMAS];
#pragma unroll
    for (int j = 0; j < DMAS; ++j) {
        a_row[j] = (wave * DMAS + j) * ROWS_PER_DMA + lane / CHUNKS;
        const int c = (lane % CHUNKS) ^ swizzle(a_row[j]);
        a_chunk[j] = (uint32_t)c * 16u;
        a_live[j] = 8 * c < K;
        // chunks past K are never fetched: zero, once, in both stages
        if (!a_live[j]) {
#pragma unroll
            for (int st = 0; st < 2; ++st) *reinterpret_cast<uint4*>(lds + st * STAGE + (wave * DMAS + j) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
        }
    }
    auto issue_a = [&](int z, int mt, uint32_t stage) __attribute__((always_inline)) {
        const uint8_t* const src = reinterpret_cast<const uint8_t*>(a_dense + (int64_t)z * gb.a) + (size_t)mt * SH_M * (size_t)K * 2;
        const int last = M - 1 - mt * SH_M;
#pragma unroll
        for (int j = 0; j < DMAS; ++j) {
            const uint32_t voff = (uint32_t)min(a_row[j], last) * (uint32_t)K * 2u + a_chunk[j];
            const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_addr + stage * STAGE + (uint32_t)(wave * DMAS + j) * 1024u));
            if (a_live[j]) dma_1kb(dst, voff, src);        // (at least a quarter of the lanes)
        }
    };
    // first tile; (z, tile_n, mt) advance with t
    const uint32_t column = t0 / (uint32_t)m_tiles;
    int mt = __builtin_amdgcn_readfirstlane((int)(t0 - column * (uint32_t)m_tiles));
    int z = __builtin_amdgcn_readfirstlane((int)(column / (uint32_t)n_tiles));
    int tile_n = __builtin_amdgcn_readfirstlane((int)(column % (uint32_t)n_tiles));
    issue_a(z, mt, 0);

    // fragment of the 16-k step q: chunk 2 q + lane / 32 of row 32 wave_m + lane % 32, i.e. f_off with chunk bits 1.. flipped by q
    const uint32_t f_off = (uint32_t)(32 * wave_m + r32) * ROW + (uint32_t)((g2 ^ swizzle(r32)) * 16);
    uint8_t* const out = lds + 2 * STAGE + wave * SH_STAGE_OUT;
    // whole 16-byte runs: every row piece starts and ends on a 16-byte boundary
    const bool vec = (N * ESZ) % 16 == 0 && (reinterpret_cast<uintptr_t>(y_all) & 15) == 0 && (gb.y & 15) == 0;
    // rows of whole 128-byte lines go past the caches (the outputs are not read here); others leave half-filled lines, which
    // the L2 puts together with the neighbours' halves
    const bool lines = vec && (N * ESZ) % 128 == 0 && (reinterpret_cast<uintptr_t>(y_all) & 127) == 0 && (gb.y & 127) == 0;

    bf16x8 wf[2][Q];                                       // W, composed: rows n0 + 32 j + lane % 32, k 16 q + 8 (lane / 32) ..
    bool new_column = true;
    for (uint32_t t = t0; t < t1; ++t) {
        const uint32_t stage = (t - t0) & 1u;
        const int n0 = tile_n * SH_N + wave_n * 64;        // the wavefront's first column
        if (new_column) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int64_t n = min(n0 + 32 * j + r32, N - 1);
                const uint8_t* const wr = w_elements + (int64_t)z * gb.we + n * K + 8 * g2;
                const uint8_t* const sr = w_scales + (int64_t)z * gb.ws + n * (K / 32);
                uint2 raw[Q];
                uint32_t sc[Q / 2];
#pragma unroll
                for (int q = 0; q < Q; ++q) raw[q] = 16 * q < K ? *reinterpret_cast<const uint2*>(wr + 16 * q) : make_uint2(0u, 0u);
#pragma unroll
                for (int b = 0; b < Q / 2; ++b) sc[b] = 32 * b < K ? sr[b] : 127u;
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    const Composer<FW> c(sc[q / 2]);
                    uint32_t o[4];
                    c.pair2(raw[q].x, o[0], o[1]);
                    c.pair2(raw[q].y, o[2], o[3]);
                    if (__builtin_amdgcn_ballot_w64(Composer<FW>::is_slow(sc[q / 2])) != 0 && Composer<FW>::is_slow(sc[q / 2])) {
                        c.pair2_slow(raw[q].x, o[0], o[1]);
                        c.pair2_slow(raw[q].y, o[2], o[3]);
                    }
                    typedef uint32_t u32v4_t __attribute__((ext_vector_type(4)));
                    wf[j][q] = __builtin_bit_cast(bf16x8, u32v4_t{o[0], o[1], o[2], o[3]});
                }
            }
        }
        // this wavefront's DMAs of this A tile are older than the last tile's stores; LDS reads of the last tile are done
        if (vec && !new_column) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(STORES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int mt_now = mt;
        uint8_t* const y_base = static_cast<uint8_t*>(y_all) + (int64_t)z * gb.y;
        new_column = ++mt == m_tiles;
        if (new_column) {
            mt = 0;
            if (++tile_n == n_tiles) { tile_n = 0; ++z; }
        }
        mt = __builtin_amdgcn_readfirstlane(mt);           // (uniform; said again for the scalar operands of the DMA)
        z = __builtin_amdgcn_readfirstlane(z);
        if (t + 1 < t1) issue_a(z, mt, stage ^ 1);
        floatx16 acc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[j][v] = 0.0f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const bf16x8 af = *reinterpret_cast<const bf16x8*>(lds + stage * STAGE + (f_off ^ (32u * q)));
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[0][q], af, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[1][q], af, acc[1], 0, 0, 0);
        }
        // lane holds y[m][n .. n + 3] with m = lane % 32, n = 32 j + 8 g + 4 (lane / 32) of the wavefront's 32 x 64 outputs
        const int m_first = mt_now * SH_M + 32 * wave_m;
        uint8_t* const y_tile = y_base + (size_t)m_first * (size_t)N * ESZ;
        const int64_t rows_left = M - m_first;
        // (a tile whose rows are all past M stores nothing: zero bytes are in bounds)
        const uint32_t y_bytes = rows_left > 0 ? (uint32_t)min(rows_left, (int64_t)32) * (uint32_t)N * ESZ : 0u;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(y_tile, (short)0, (int)y_bytes, 0x00020000);
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
            // staging row = 128 bytes of the output row; the 16-byte piece c of row r at position c ^ ((r >> 1) & 7)
            const uint32_t o_off = (uint32_t)r32 * 128u + (uint32_t)((r32 >> 1) & 7) * 16u;
#pragma unroll
            for (int jj = 0; jj < 2 / PASSES; ++jj) {
                const int j = PASSES == 2 ? p : jj;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    if constexpr (DT_OUT == F32) {
                        *reinterpret_cast<float4*>(out + (o_off ^ (32u * g + 16u * g2))) =
                            make_float4(acc[j][4 * g], acc[j][4 * g + 1], acc[j][4 * g + 2], acc[j][4 * g + 3]);
                    } else {
                        uint2 v;
                        if (DT_OUT == BF16) v = make_uint2(cvt_pk_bf16(acc[j][4 * g], acc[j][4 * g + 1]), cvt_pk_bf16(acc[j][4 * g + 2], acc[j][4 * g + 3]));
                        else v = make_uint2(f32_bits_to_half_bits(f32_bits(acc[j][4 * g])) | (f32_bits_to_half_bits(f32_bits(acc[j][4 * g + 1])) << 16),
                                            f32_bits_to_half_bits(f32_bits(acc[j][4 * g + 2])) | (f32_bits_to_half_bits(f32_bits(acc[j][4 * g + 3])) << 16));
                        *reinterpret_cast<uint2*>(out + (o_off ^ (64u * j + 16u * g)) + 8 * g2) = v;
                    }
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the wavefront's own writes: no other wavefront uses this piece)
            const int col0 = n0 + (PASSES == 2 ? 32 * p : 0);    // column of the staging row's first byte
            if (vec) {
                typedef uint32_t u32v4_t __attribute__((ext_vector_type(4)));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = 8 * i + (lane >> 3), c = lane & 7;
                    const u32v4_t v = *reinterpret_cast<const u32v4_t*>(out + row * 128 + ((c ^ ((row >> 1) & 7)) * 16));
                    const int col = col0 + c * (16 / ESZ);
                    const uint32_t off = col < N ? ((uint32_t)row * (uint32_t)N + (uint32_t)col) * ESZ : 0xFFFFFFF0u;   // past the end: dropped
                    if (lines) __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)off, 0, 2 /* nt */);
                    else __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, (int)off, 0, 0);
                }
            } else {
                constexpr int COLS = 128 / ESZ;                  // columns of a staging row
                const int steps = (int)((min(rows_left, (int64_t)32) * COLS + 63) / 64);   // rows there are (rows past M: none, also below zero)
#pragma unroll 1
                for (int i = 0; i < steps; ++i) {
                    const int row = i * 64 / COLS + (COLS == 32 ? g2 : 0), b = (lane % COLS) * ESZ;
                    const int col = col0 + lane % COLS;
                    const uint8_t* const s = out + row * 128 + (((b >> 4) ^ ((row >> 1) & 7)) * 16) + (b & 15);
                    if (row < rows_left && col < N) {
                        if (ESZ == 4) *reinterpret_cast<uint32_t*>(y_tile + ((size_t)row * N + col) * 4) = *reinterpret_cast<const uint32_t*>(s);
                        else *reinterpret_cast<uint16_t*>(y_tile + ((size_t)row * N + col) * 2) = *reinterpret_cast<const uint16_t*>(s);
                    }
                }
            }
            asm volatile("" ::: "memory");
        }
    }
}

template <class FW, int DT_OUT>
int launch_gemm_short_k(const GemmArgs& g) {
    const int cus = device_cu_count();
    if (cus <= 0) return fail(ERR_RUNTIME, "cannot read the compute-unit count of the current device");
    const int n_tiles = (g.N + SH_N - 1) / SH_N, m_tiles = (g.M + SH_M - 1) / SH_M;
    // two workgroups per CU, each with an equal run of tiles
    const int64_t items = (int64_t)g.batches * n_tiles * m_tiles;
    if (items > 0x7FFFFFFFll) return fail(ERR_UNSUPPORTED, "too many tiles for one launch");
    const unsigned grid = (unsigned)((std::min<int64_t>(items, 2ll * cus) + 7) / 8 * 8);
    auto kern = g.K <= 64 ? mxfp_gemm_short_k_kernel<FW, DT_OUT, 64> : mxfp_gemm_short_k_kernel<FW, DT_OUT, 128>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, g.stream, static_cast<const uint16_t*>(g.a_dense), g.w_scales, g.w_elements, g.y, g.M,
                       g.N, g.K, n_tiles, m_tiles, (uint32_t)(items / grid), (uint32_t)(items % grid), g.batch);
    return check_launch("mxfp_gemm");
}

}  // namespace mase
