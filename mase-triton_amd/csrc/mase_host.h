// Host-side helpers shared by the C-ABI entry points: error reporting and argument checks.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <algorithm>
#include <atomic>
#include <string>

#include "mase_device.h"

namespace mase {

enum Status : int { OK = 0, ERR_INVALID = -1, ERR_UNSUPPORTED = -2, ERR_RUNTIME = -3 };

std::string& last_error();  // thread-local message of the most recent failure

inline int fail(int code, const std::string& msg) {
    last_error() = msg;
    return code;
}

inline int check_launch(const char* what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(ERR_RUNTIME, std::string(what) + ": " + hipGetErrorString(e));
    return OK;
}

// A kernel that uses more than 64 KB of dynamic LDS has to be given the limit once on every device it runs on (the
// attribute belongs to the function as loaded on the current device).  `done` is the call site's record: bit d = set on
// device d; devices past 63 set it on every launch.  Safe from several threads (setting it twice is harmless).
inline int allow_dynamic_lds(const void* kern, int bytes, std::atomic<uint64_t>& done) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail(ERR_RUNTIME, std::string("hipGetDevice: ") + hipGetErrorString(e));
    const uint64_t bit = dev >= 0 && dev < 64 ? uint64_t(1) << dev : 0;
    if (bit && (done.load(std::memory_order_relaxed) & bit)) return OK;
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return fail(ERR_RUNTIME, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
    done.fetch_or(bit, std::memory_order_relaxed);
    return OK;
}

// compute units of the current device (at least 8), or -1
inline int device_cu_count() {
    static std::atomic<int> cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return -1;
    const bool cached = dev >= 0 && dev < 64;
    int n = cached ? cus[dev].load(std::memory_order_relaxed) : 0;
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return -1;
        n = n > 8 ? n : 8;
        if (cached) cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; }

inline int check_minifloat_fmt(int E, int M, int rm) {
    if (E < 1 || M < 1 || E + M >= 16) return fail(ERR_INVALID, "minifloat format needs exp_bits >= 1, frac_bits >= 1, exp_bits + frac_bits < 16");
    if (rm < RN || rm > RZ) return fail(ERR_INVALID, "round_mode must be 0 (rn), 1 (ru), 2 (rd) or 3 (rz)");
    return OK;
}

inline int check_mxfp_fmt(int E, int M, int rm, int64_t n, int block) {
    const bool legal = (E == 4 && M == 3) || (E == 5 && M == 2) || (E == 2 && M == 3) || (E == 3 && M == 2) ||
                       (E == 2 && M == 1);
    if (!legal) return fail(ERR_INVALID, "MXFP element (exp_bits, frac_bits) must be one of (4,3) (5,2) (2,3) (3,2) (2,1)");
    if (rm < RN || rm > RZ) return fail(ERR_INVALID, "round_mode must be 0 (rn), 1 (ru), 2 (rd) or 3 (rz)");
    if (block < 1) return fail(ERR_INVALID, "block_size must be positive");
    if (n < 0 || n % block != 0) return fail(ERR_INVALID, "element count must be a non-negative multiple of block_size");
    return OK;
}

inline int check_dtype(int dt, const char* which) {
    if (dt != F32 && dt != F16 && dt != BF16) return fail(ERR_INVALID, std::string(which) + " dtype must be 0 (f32), 1 (f16) or 2 (bf16)");
    return OK;
}

inline int dtype_size(int dt) { return dt == F32 ? 4 : 2; }

// Extract down the rows of `columns` columns and nkb k-blocks in tiles of 64 columns (one wavefront per tile and k-block)?  A tile that
// its columns do not fill costs a whole one, which shows once there are more wavefronts than the chip has room to overlap: from
// then on the kernel whose lanes are blocks of any column.  fp32, tiles / other kernel, us, at 512, 2048, 8192 and 32768 k-blocks: 1 column
// 4.2 / 6.8, 5.4 / 6.8, 13.9 / 6.9, 48 / 7.0; 16 columns 4.2 / 4.1, 5.5 / 4.3, 14.6 / 6.0, 49 / 24 (fp16 53 / 18); 48 columns 4.4 / 4.4,
// 5.9 / 6.2, 16.4 / 15.5; 65 columns 4.3 / 4.8, 8.9 / 7.8, 27.3 / 24.8; 96 columns 4.4 / 5.0, 9.1 / 9.4, 28.4 / 28.5 (fp16 28.8 / 24.4); 97 columns
// 4.4 / 5.2, 9.3 / 10.7, 28.8 / 32.6 (fp16 29.1 / 27.6); fp32 129 columns 22.2 / 23.9 at 4096, fp16 22.4 / 20.2.  Fuller tiles are ahead at every size but the smallest, where they are level.
// The same for the four k-blocks of a workgroup: with 262144 columns 14.8 / 9.6 at one k-block (fp16 14.5 / 9.5), and 21.1 / 20.4 (21.2 / 19.3)
// at two; 29.8 / 26.2 (28.9 / 19.9) at five and 131072; at 65536 columns of one or two k-blocks 7.6 / 8.2 and 11.2 / 12.6.
inline bool strided_column_tiles(int64_t columns, int64_t nkb, int element_bytes) {
    const int64_t tiles = (columns + 63) / 64, waves = tiles * nkb, groups = (nkb + 3) / 4;
    if (waves >= 2048 && columns * 2 <= tiles * 64) return false;
    if (waves >= 4096 && columns * 8 <= tiles * 64 * (element_bytes == 4 ? 5 : 6)) return false;
    return tiles * groups < 2048 || nkb * 8 > groups * 4 * 5;
}

// The same for the kernel that takes two columns of 16-bit elements to a lane, 128 columns and four k-blocks to a workgroup.  bf16, against the
// kernel that stores a column's codes by itself, us: 2976 x 4096 11.2 / 12.6, 65536 x 200 12.5 / 15.6, 1024 x 2050 4.8 / 6.1; tiles that the columns or k-blocks
// leave half empty cost once there are many: 160 x 65536 (five k-blocks) 13.5 / 10.8, 32 x 262144 level without it.  fp16, against one column to a lane:
// 2976 x 4096 12.5 / 14.7, 65536 x 200 13.6 / 17.5, 256 x 9000 5.2 / 6.0; with fewer wavefronts the other kernel's shorter lanes are ahead: 96 x 14336 4.9 / 4.5,
// 64 x 1000 4.6 / 4.2, 64 matrices of 512 x 64 5.3 / 4.9.
// Rows (the inner axis) of a few columns behind a longer outer axis: a load then takes pieces of many matrices.  bf16 rows of fewer than 80 columns:
// filled tiles are behind (1000 matrices of 2080 x 2 15.5 / 10.4, 32 of 87360 x 6 26.2 / 19.0, 128 of 10912 x 12 20.0 / 17.0, 3 of 2048 or 8192 x 32 7.3 / 6.8
// and 17.7 / 17.1; at best 3 % ahead), a few columns in all are what the other kernel leaves its lanes idle for (65536 x 2 4.1 / 6.9, 8 x 4096 x 8 4.4 /
// 4.8) until their wavefronts are many (36832 x 64 6.4 / 5.7, 11 of 27776 x 12 8.6 / 6.7).  fp16: rows of 4 (32 matrices of 32768 or 131072: 9.2 / 7.5, 26.9 /
// 19.6) and 12 columns (9.1 / 8.4, level when many); 2, 6, 8 and longer ones are ahead (10.6 / 12.3, 6.8 / 7.3).
inline bool strided_pair_tiles(int64_t inner, int64_t columns, int64_t nkb, bool bf16) {
    const int64_t tiles = (columns + 127) / 128, groups = (nkb + 3) / 4, waves = tiles * groups * 4;
    const bool filled = columns * nkb * 10 >= tiles * 128 * groups * 4 * 7;
    if (!bf16) return filled && waves > 512 && inner != 4 && inner != 12;
    return inner < 80 ? !filled && waves <= 1024 : filled || waves < 2048;
}

// Calls fn(format object): a compile-time format for the five round-to-nearest finite
// presets, the run-time one otherwise.
template <class Fn>
inline int dispatch_fmt(int E, int M, int fin, int rm, Fn&& fn) {
    if (fin && rm == RN) {
        if (E == 4 && M == 3) return fn(SFmt<4, 3>{});
        if (E == 5 && M == 2) return fn(SFmt<5, 2>{});
        if (E == 2 && M == 3) return fn(SFmt<2, 3>{});
        if (E == 3 && M == 2) return fn(SFmt<3, 2>{});
        if (E == 2 && M == 1) return fn(SFmt<2, 1>{});
    }
    return fn(DFmt{E, M, fin, rm});
}

template <int V> struct IntC { static constexpr int value = V; };

template <class Fn>
inline int dispatch_dtype(int dt, Fn&& fn) {
    switch (dt) {
        case F32: return fn(IntC<F32>{});
        case F16: return fn(IntC<F16>{});
        default: return fn(IntC<BF16>{});
    }
}

}  // namespace mase
