// Products of a short contraction that quantise on the way in:  y[M,N] = Q(A)[M,K] * W[N,K]^T for K <= 128, bf16 in and out, one or
// many products per launch: attention scores, batch x heads products of queries against keys with K = the head dimension.  A is
// dense bf16 and goes through the MXFP quantise-dequantise (blocks of 32 along K, exact in bf16) in registers; W is bf16 that is
// quantised already or goes the same way as A.
//
// The outputs are what there is to move (64 products of 1000 x 1000 x 128: 128 of 161 MB), so the kernel is built around
// how they leave:
//   * a workgroup owns 128 rows of A (32 per wavefront, quantised once, fragments in registers) and walks along the rows of W, 64
//     at a time, so a row of y is written from left to right by one wavefront;
//   * rows of y need not start at a 128-byte line (2000-byte rows of 1000 columns): a step does not store the 64 columns it has
//     computed but the 64 columns that end at the last line boundary it has passed, the rest staying in LDS for the next step.  All
//     stores but the first and last of a row are whole lines, past the caches.  Stored tile by tile instead, every row piece
//     begins and ends inside a line, the caches fill with half-written lines and the operands wait behind their write-back;
//   * panels start at different columns and wrap around, so that the chip does not write one column of every row at a time: 32
//     products of 2048 x 2048 (4096-byte rows) 92 us without, 75 with;
//   * W tiles of 64 x K go global -> LDS by DMA, two steps ahead, and a wavefront waits for its share with a count that leaves its
//     latest stores out; a panel first asks for its share of W at once, so that the steps find W in the L2 (58 us without, 47 with);
//   * or W comes raw through four more wavefronts that quantise it (a few panels of A: once for each of them costs less than a pass
//     over W and its launch);
//   * wavefront-private staging, one barrier per step, two workgroups per CU.
// The steps of all panels are dealt to the workgroups in equal contiguous runs; those of one product share an XCD's L2.
//
// Measured, E4M3, other operands and outputs on every call, everything included, against the two casts and the kernels of
// gemm_short_k.h: 64 products of 1000 x 1000 x 128 47 us (34 without the pass over W) against 62; 32 of 2048 x 2048 x 128 75 against
// 106; 32 of 1464 x 1464 x 64 36 against 48; W quantised on the way in: 32 of 512 x 512 x 128 14.6 against 30, 128 of 40 x 2048 x 128
// 32 against 54, 64 of 64 rows 4.4 against 8.4.  What bounds the large ones: operands are read before the first store can leave
// (8 us), a step takes 0.9 us of LDS reads, MFMAs and conversions (24 us with the stores left out), y alone is 20 us of writes.
#pragma once
#include "gemm_impl.h"
#include "mxfp_bf16.h"

namespace mase {

constexpr int SCO_M = 128, SCO_N = 64, SCO_MAX_K = 128;
constexpr int SCO_STAGE = 2 * 32 * 128;                  // a wavefront's staging: two chunks of 32 rows x 64 outputs
constexpr int SCO_TILES = 3;                             // W tiles in LDS
template <int KP> constexpr int sco_lds_bytes() { return SCO_TILES * SCO_N * 2 * KP + 4 * SCO_STAGE; }
template <bool QW> constexpr int sco_threads() { return QW ? 512 : 256; }

struct ScoresArgs {
    const uint16_t* a; const uint16_t* w; uint16_t* y;
    int M, N, K, n_steps, panels;
    uint32_t per_run, longer_runs;                        // steps of a workgroup's run; the first `longer_runs` have one more
    int64_t a_stride, w_stride, y_stride;                 // elements between products
};

// QA / QW: quantise A / W in format F on the way in.  KP: the K the loops are built for (64 or 128); a smaller K is filled with zeros.
// Wavefronts 0 - 3 multiply and store, the others (one, or four that quantise) bring W.  A wavefront's memory operations complete
// in order, and a store takes microseconds to be acknowledged while the memory is busy writing: a wavefront that stored and
// waited for loads as well would wait for its stores.  (The builds of KP = 128 that quantise W do: 128 registers are all that four wavefronts
// per SIMD leave them, and 72 - 80 bytes per lane go through scratch.  They wait with the compiler's counts only; mase_hip_mxfp_scores_plan has their times.)
template <class F, bool QA, bool QW, int KP>
__global__ __launch_bounds__(sco_threads<QW>()) __attribute__((amdgpu_waves_per_eu(QW ? 4 : 2))) void mxfp_scores_kernel(const ScoresArgs p) {
    constexpr int Q = KP / 16;                             // 16-k steps
    constexpr int ROW = 2 * KP, CHUNKS = ROW / 16;         // bytes and 16-byte pieces of an operand row in LDS
    constexpr int TILE = SCO_N * ROW;                      // one W tile
    constexpr int PIECES = TILE / 1024;                    // 1 KB pieces of it
    constexpr int ROWS_PER_KB = 1024 / ROW;
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];   // the W tiles, the staging of wavefronts 0 - 3
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = p.M, N = p.N, K = p.K, n_steps = p.n_steps;
    // workgroups are dealt to the 8 XCDs in turn; XCD x takes the x-th eighth of the runs (the grid is a multiple of 8)
    const uint32_t run = (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    const uint32_t t0 = run * p.per_run + min(run, p.longer_runs), t1 = t0 + p.per_run + (run < p.longer_runs ? 1u : 0u);
    if (t0 >= t1) return;
    const uint32_t panel0 = t0 / (uint32_t)n_steps;
    int step = __builtin_amdgcn_readfirstlane((int)(t0 - panel0 * (uint32_t)n_steps));
    int z = __builtin_amdgcn_readfirstlane((int)(panel0 / (uint32_t)p.panels));
    int panel = __builtin_amdgcn_readfirstlane((int)(panel0 % (uint32_t)p.panels));
    auto advance = [&]() __attribute__((always_inline)) {
        if (++step == n_steps) {
            step = 0;
            if (++panel == p.panels) { panel = 0; ++z; }
        }
        step = __builtin_amdgcn_readfirstlane(step);
        panel = __builtin_amdgcn_readfirstlane(panel);
        z = __builtin_amdgcn_readfirstlane(z);
    };
    // Which 64 columns a step of a panel is: panels start at different places of their rows and wrap around (rows of y are N * 2 bytes
    // apart, with N a power of two all rows' pieces at one place are on the same few channels of the memory)
    auto column_step = [&](int zz, int pp, int ss) __attribute__((always_inline)) {
        const int at = ss + (int)((uint32_t)(5 * pp + 3 * zz) % (uint32_t)n_steps);
        return __builtin_amdgcn_readfirstlane(at >= n_steps ? at - n_steps : at);
    };
    // piece c of row r sits at position c ^ swizzle(r): conflict-free 128-bit fragment reads
    auto swizzle = [](int row) { return KP == 128 ? (row & 15) : ((row >> 1) & 7); };

    if constexpr (QW) {
        if (wave >= 4) {
            // four wavefronts, a quarter of the tile each, four lanes to a block; one tile ahead in registers, one in LDS
            constexpr int PER = PIECES / 4;
            const int first = (wave - 4) * PER;
            uint4 raw[PER];
            auto load = [&]() __attribute__((always_inline)) {
                const uint16_t* const src = p.w + (int64_t)z * p.w_stride;
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int row = (first + j) * ROWS_PER_KB + lane / CHUNKS, c = lane % CHUNKS;      // (rows past N re-read row N - 1)
                    raw[j] = 8 * c < K ? *reinterpret_cast<const uint4*>(src + (int64_t)min(column_step(z, panel, step) * SCO_N + row, N - 1) * K + 8 * c) : make_uint4(0, 0, 0, 0);
                }
            };
            load();
            uint32_t tile = 0;
            for (uint32_t t = t0; t < t1; ++t) {
#pragma unroll
                for (int j = 0; j < PER; ++j) {
                    const int row = (first + j) * ROWS_PER_KB + lane / CHUNKS, c = lane % CHUNKS;
                    uint32_t o[4], scale;
                    bf16_block_step<F, true>(raw[j], F{}, o, scale, 0u);
                    *reinterpret_cast<uint4*>(lds + tile * TILE + row * ROW + ((c ^ swizzle(row)) * 16)) = make_uint4(o[0], o[1], o[2], o[3]);
                }
                tile = tile == SCO_TILES - 1 ? 0 : tile + 1;
                advance();
                if (t + 1 < t1) load();
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();              // tile t is there; everyone has done with tile t - 1
                asm volatile("" ::: "memory");
            }
            return;
        }
    }
    // ---- W by DMA: four (two) pieces of 1 KB per wavefront and tile, two tiles ahead.  Lane l of a piece fills position l % CHUNKS of a
    //      row with the piece of the row that belongs there; what lies past K is never fetched: zero, once, in all tiles
    constexpr int PER = PIECES / 4;
    const uint32_t lds_addr = (uint32_t)(uintptr_t)lds;
    int w_row[PER];
    uint32_t w_piece[PER];
    int z_next = z, panel_next = panel, step_next = step;  // of the tile that is fetched next
    if constexpr (!QW) {
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            w_row[j] = (wave * PER + j) * ROWS_PER_KB + lane / CHUNKS;
            w_piece[j] = (uint32_t)((lane % CHUNKS) ^ swizzle(w_row[j])) * 8u;
            if ((int)w_piece[j] >= K) {
#pragma unroll
                for (int b = 0; b < SCO_TILES; ++b) *reinterpret_cast<uint4*>(lds + b * TILE + (wave * PER + j) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
            }
        }
    }
    auto fetch = [&](uint32_t tile) __attribute__((always_inline)) {
        const int at = column_step(z_next, panel_next, step_next);
        const uint16_t* const src = p.w + (int64_t)z_next * p.w_stride + (int64_t)at * SCO_N * K;
        const int last = N - 1 - at * SCO_N;               // rows past N re-read row N - 1
#pragma unroll
        for (int j = 0; j < PER; ++j) {
            const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_addr + tile * TILE + (uint32_t)(wave * PER + j) * 1024u));
            if ((int)w_piece[j] < K) dma_1kb(dst, ((uint32_t)min(w_row[j], last) * (uint32_t)K + w_piece[j]) * 2u, src);     // (at least a quarter of the lanes)
        }
        if (++step_next == n_steps) {
            step_next = 0;
            if (++panel_next == p.panels) { panel_next = 0; ++z_next; }
        }
        step_next = __builtin_amdgcn_readfirstlane(step_next);
        panel_next = __builtin_amdgcn_readfirstlane(panel_next);
        z_next = __builtin_amdgcn_readfirstlane(z_next);
    };
    if constexpr (!QW) {
        fetch(0);
        if (t0 + 1 < t1) fetch(1);
    }

    const int g2 = lane >> 5, r32 = lane & 31;
    uint8_t* const stage = lds + SCO_TILES * TILE + wave * SCO_STAGE;
    bf16x8 af[Q];                                          // A, quantised: row 32 wave + lane % 32 of the panel, k 16 q + 8 (lane / 32) ..
    int at = column_step(z, panel, step), first = at;      // this step's columns, and where the run of columns that it belongs to began
    bool new_panel = true;
    // The pieces of y that the lane stores, row 8 i + lane / 8 each: step `at` sends piece 8 at + (lane & 7) - (where the row starts in
    // its line, in pieces) of the row, which sits in chunk at or at - 1 of the staging
    typedef uint32_t u32v4_t __attribute__((ext_vector_type(4)));
    int piece[4];                                          // of step 0: -7 .. 7
    uint32_t y_off[4], s_off[4];                           // step 1's offset in y (rows past M: NO_ROW) and step 0's in the staging (odd steps: the other chunk)
    constexpr uint32_t NO_ROW = 0xFFFFFFF0u;               // past the end of every descriptor: dropped
    // Descriptors of the wavefront's rows of y.  `whole`: for the steps inside a row, whose pieces are all there (the step's offset comes
    // on top of what is checked against its size); `rsrc`: exact; `none`: drops everything
    __amdgpu_buffer_rsrc_t rsrc, whole, none;
    auto take = [&](u32v4_t (&v)[4], uint32_t chunk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const u32v4_t*>(stage + (s_off[i] ^ chunk));
    };
    // what of columns' step `which` lies in lo <= column < hi, at once
    auto flush = [&](int which, int lo, int hi) __attribute__((always_inline)) {
        u32v4_t v[4];
        take(v, (uint32_t)(which & 1) * 4096u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int col = 8 * (8 * which + piece[i]);
            const uint32_t off = col >= lo && col < hi && y_off[i] != NO_ROW ? y_off[i] + 128u * (uint32_t)(which - 1) : NO_ROW;
            __builtin_amdgcn_raw_buffer_store_b128(v[i], rsrc, (int)off, 0, 0);
        }
    };
    // staging row = 128 bytes of a row of the tile; the 16-byte piece c of row r at position c ^ ((r >> 1) & 7)
    const uint32_t o_off = (uint32_t)r32 * 128u + (uint32_t)((r32 >> 1) & 7) * 16u + 8u * g2;
    const uint32_t frag = (uint32_t)r32 * ROW + (uint32_t)((g2 ^ swizzle(r32)) * 16);
    uint32_t tile = 0;
    int landed = 0;                                        // tiles from t on that are known to be there
    for (uint32_t t = t0; t < t1; ++t) {
        if (new_panel) {
            // the wavefront's 32 rows of A, through its own staging: rows past M re-read row M - 1
            constexpr int LOADS = 32 / ROWS_PER_KB;
            const int m_first = panel * SCO_M + 32 * wave;
            const uint16_t* const src = p.a + (int64_t)z * p.a_stride;
            uint4 raw[LOADS];
#pragma unroll
            for (int j = 0; j < LOADS; ++j) {
                const int row = j * ROWS_PER_KB + lane / CHUNKS, c = lane % CHUNKS;
                raw[j] = 8 * c < K ? *reinterpret_cast<const uint4*>(src + (int64_t)min(m_first + row, M - 1) * K + 8 * c) : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int j = 0; j < LOADS; ++j) {
                const int row = j * ROWS_PER_KB + lane / CHUNKS, c = lane % CHUNKS;
                uint32_t o[4] = {raw[j].x, raw[j].y, raw[j].z, raw[j].w}, scale;
                if constexpr (QA) bf16_block_step<F, true>(raw[j], F{}, o, scale, 0u);
                *reinterpret_cast<uint4*>(stage + row * ROW + ((c ^ swizzle(row)) * 16)) = make_uint4(o[0], o[1], o[2], o[3]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the wavefront's own writes)
#pragma unroll
            for (int q = 0; q < Q; ++q) af[q] = *reinterpret_cast<const bf16x8*>(stage + (frag ^ (32u * q)));
            uint16_t* const y_rows = p.y + (int64_t)z * p.y_stride + (int64_t)m_first * N;
            const int rows = min(max(M - m_first, 0), 32);
            rsrc = __builtin_amdgcn_make_buffer_rsrc(y_rows, (short)0, (int)((uint32_t)rows * (uint32_t)N * 2u), 0x00020000);
            whole = __builtin_amdgcn_make_buffer_rsrc(y_rows, (short)0, (int)((uint32_t)rows * (uint32_t)N * 2u + 256u), 0x00020000);
            none = __builtin_amdgcn_make_buffer_rsrc(y_rows, (short)0, 0, 0x00020000);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t row = 8u * i + (uint32_t)(lane >> 3);
                piece[i] = (lane & 7) - (int)(((uint32_t)(reinterpret_cast<uintptr_t>(y_rows) >> 4) + row * (uint32_t)(N >> 3)) & 7u);
                y_off[i] = (int)row < rows ? (row * (uint32_t)N + (uint32_t)(8 * piece[i])) * 2u + 128u : NO_ROW;
                s_off[i] = (uint32_t)((piece[i] >> 3) & 1) * 4096u + row * 128u + (((uint32_t)(piece[i] & 7) ^ ((row >> 1) & 7u)) * 16u);
            }
            first = at;
            landed = 2;
        }
        if constexpr (QW) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
            // This wavefront's pieces of tile t have landed: they are older than A, or than the four stores of step t - 2, the pieces of
            // tile t + 1 and the four stores of step t - 1, which may still be on their way (a store takes microseconds to be
            // acknowledged while the memory is busy writing)
            if (landed > 0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            else if (t + 1 < t1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(8 + PER) : "memory");
            else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)" ::: "memory");
            landed = landed > 0 ? landed - 1 : 0;
        }
        __builtin_amdgcn_s_barrier();                      // tile t is there; everyone has done with tile t - 1
        asm volatile("" ::: "memory");
        if constexpr (!QW) {
            const uint32_t free = tile == 0 ? SCO_TILES - 1 : tile - 1;
            if (new_panel && K == KP) {                    // (a shorter K has zeros in the tiles that have to stay)
                // this panel's share of the product's W into the L2, all at once (what arrives lands in the tile that is fetched next)
                const uint32_t w_bytes = (uint32_t)N * (uint32_t)K * 2u;
                const uint32_t share = ((w_bytes + 4095u) / 4096u + (uint32_t)p.panels - 1u) / (uint32_t)p.panels;
                const uint32_t dst = (uint32_t)__builtin_amdgcn_readfirstlane((int)(lds_addr + free * TILE + (uint32_t)(wave * PER) * 1024u));
                const uint8_t* const src = reinterpret_cast<const uint8_t*>(p.w + (int64_t)z * p.w_stride);
                for (uint32_t i = 0; i < min(share, 16u); ++i)
                    dma_1kb(dst, min(((uint32_t)panel * share + i) * 4096u + (uint32_t)wave * 1024u + (uint32_t)lane * 16u, w_bytes - 16u), src);
            }
            if (t + 2 < t1) fetch(free);
        }
        // the step before leaves while this one is multiplied (a row's first step has left by itself, see below)
        // Fragments of W are asked for up to three 16-k steps ahead, the pieces of y beside the first of them; their order is pinned (left to
        // itself the compiler asks for each fragment right before it is multiplied and the matrix unit waits for the LDS).
        const bool behind = at - 1 > first;                  // (so at - 2 >= 0)
        const uint8_t* const w_tile = lds + tile * TILE;
        const uint32_t other = (uint32_t)((at - 1) & 1) * 4096u;
        u32v4_t v[4];
        constexpr int AHEAD = QW ? 1 : 3, RING = AHEAD + 1;
        bf16x8 wf[RING][2];
        auto read = [&](int q) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; ++j) wf[q % RING][j] = *reinterpret_cast<const bf16x8*>(w_tile + j * 32 * ROW + (frag ^ (32u * q)));
        };
#pragma unroll
        for (int q = 0; q < AHEAD; ++q) read(q);
        __builtin_amdgcn_sched_barrier(0);
        floatx16 acc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[j][e] = 0.0f;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if (q + AHEAD < Q) read(q + AHEAD);
            if (q < 4) v[q] = *reinterpret_cast<const u32v4_t*>(stage + (s_off[q] ^ other));
            if (q >= Q - 4)
                __builtin_amdgcn_raw_buffer_store_b128(v[q - (Q - 4)], behind ? whole : none, (int)y_off[q - (Q - 4)], 128 * (at - 2), 2 /* past the caches */);
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[q % RING][j], af[q], acc[j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        // lane holds y[m][n .. n + 3] with m = lane % 32, n = 32 j + 8 g + 4 (lane / 32) of the wavefront's 32 x 64 outputs
        uint8_t* const chunk = stage + (at & 1) * 4096;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<uint2*>(chunk + (o_off ^ (64u * j + 16u * g))) =
                    make_uint2(cvt_pk_bf16(acc[j][4 * g], acc[j][4 * g + 1]), cvt_pk_bf16(acc[j][4 * g + 2], acc[j][4 * g + 3]));
        const bool ends = at + 1 == n_steps || step + 1 == n_steps || t + 1 == t1;
        if (at == first || ends) {                   // (the pieces at the ends of a row share their lines with the rows beside it)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the wavefront's own writes: no other wavefront uses this piece)
            const int lo = SCO_N * first, hi = min(N, SCO_N * (at + 1));
            flush(at, lo, hi);
            if (ends) flush(at + 1, lo, hi);               // what is left behind the row's last line boundary
        }
        asm volatile("" ::: "memory");
        tile = tile == SCO_TILES - 1 ? 0 : tile + 1;
        advance();
        new_panel = step == 0;
        at = at + 1 == n_steps || new_panel ? column_step(z, panel, step) : at + 1;
        first = at == 0 ? 0 : first;                        // (a new panel sets it)
    }
}

template <class F, bool QA, bool QW>
int launch_scores(ScoresArgs p, int batches, hipStream_t s) {
    const int cus = device_cu_count();
    if (cus <= 0) return fail(ERR_RUNTIME, "cannot read the compute-unit count of the current device");
    p.n_steps = (p.N + SCO_N - 1) / SCO_N;
    p.panels = (p.M + SCO_M - 1) / SCO_M;
    const int64_t steps = (int64_t)batches * p.panels * p.n_steps;
    if (steps > 0x7FFFFFFFll) return fail(ERR_UNSUPPORTED, "too many tiles for one launch");
    // two workgroups per CU, each with an equal run of steps
    const unsigned grid = (unsigned)((std::min<int64_t>(steps, 2ll * cus) + 7) / 8 * 8);
    p.per_run = (uint32_t)(steps / grid);
    p.longer_runs = (uint32_t)(steps % grid);
    const bool k64 = p.K <= 64;
    auto kern = k64 ? mxfp_scores_kernel<F, QA, QW, 64> : mxfp_scores_kernel<F, QA, QW, 128>;
    const int lds_bytes = k64 ? sco_lds_bytes<64>() : sco_lds_bytes<128>();
    static std::atomic<uint64_t> allowed[2] = {{0}, {0}};
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_bytes, allowed[k64])) return rc;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(sco_threads<QW>()), lds_bytes, s, p);
    return check_launch("mxfp_scores");
}

}  // namespace mase
