"""The rules by which a launcher picks a kernel, asked on the CPU through the test helper library (the launchers call the same functions)."""
import ctypes
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def lib():
    path = os.path.join(ROOT, "mase-triton_amd", "mase_hip", "lib", "libmase_bench.so")
    assert os.path.exists(path), "libmase_bench.so is not built (python mase-triton_amd/build.py)"
    return ctypes.CDLL(path)


def column_tiles(lib, columns, nkb, element_bytes):
    lib.mase_bench_strided_column_tiles.argtypes = [ctypes.c_int64, ctypes.c_int64, ctypes.c_int]
    return bool(lib.mase_bench_strided_column_tiles(columns, nkb, element_bytes))


@pytest.mark.parametrize("element_bytes", [2, 4])
def test_few_columns_do_not_go_in_column_tiles(lib, element_bytes):
    for columns in (1, 3, 8, 16, 31, 32):           # wavefronts at most half full: one per k-block
        assert column_tiles(lib, columns, 2047, element_bytes)
        assert not column_tiles(lib, columns, 2048, element_bytes) and not column_tiles(lib, columns, 1 << 20, element_bytes)
    for columns in (33, 40):                        # five eighths
        assert column_tiles(lib, columns, 4095, element_bytes) and not column_tiles(lib, columns, 4096, element_bytes)
    for columns in (65, 80):                        # two wavefronts per k-block
        assert column_tiles(lib, columns, 2047, element_bytes) and not column_tiles(lib, columns, 2048, element_bytes)
    for columns in (41, 48, 96, 129):               # up to three quarters: by the element's size
        assert column_tiles(lib, columns, 1 << 16, element_bytes) == (element_bytes == 4)
    for columns in (49, 64, 97, 128, 193, 1001, 4096, 1 << 20):
        assert column_tiles(lib, columns, 3, element_bytes) and column_tiles(lib, columns, 1 << 20, element_bytes)


def test_many_columns_of_one_or_two_blocks_do_not_go_in_column_tiles(lib):
    for nkb in (1, 2):                              # of the four k-blocks of a workgroup
        assert column_tiles(lib, 1 << 16, nkb, 4) and not column_tiles(lib, 1 << 17, nkb, 4)
    assert column_tiles(lib, 1 << 15, 5, 2) and not column_tiles(lib, 1 << 16, 5, 2)      # five of eight
    for nkb in (3, 4, 6, 7, 8, 9, 93):
        assert column_tiles(lib, 1 << 20, nkb, 2)


def short_k(lib, M, N, K, batches=1):
    lib.mase_bench_short_k.argtypes = [ctypes.c_int64] * 4
    return bool(lib.mase_bench_short_k(M, N, K, batches))


def test_few_rows_of_a_short_contraction_stay_on_the_weight_streaming_kernels(lib):
    for M, most in ((1, 24576), (16, 24576), (17, 18432), (32, 18432), (33, 14336), (64, 14336)):
        assert not short_k(lib, M, 32, 128) and not short_k(lib, M, most, 128)
        assert not short_k(lib, M, 1024, 128, most // 1024)
        assert short_k(lib, M, most + 32, 128) and short_k(lib, M, 1024, 128, most // 1024 + 1)     # rows of W of all products
        assert short_k(lib, M, 4096, 64)                                    # those kernels take whole 128-k steps
    assert not short_k(lib, 8, 48, 128) and short_k(lib, 9, 12304, 128) and short_k(lib, 40, 8208, 128)   # 16-row groups up to 12288 / 8192 only
    assert short_k(lib, 65, 4096, 128) and short_k(lib, 1000, 1000, 128, 64)
    assert not short_k(lib, 4096, 4096, 160)


def test_full_rounds_of_large_tiles_stay_on_the_kernel_of_large_tiles(lib):
    for M, N in ((1024, 14336), (512, 28672), (3000, 4096), (16384, 1024), (16384, 4096), (16384, 14336), (1000, 12288)):   # 160 tiles of 512 x 128 or more
        assert not short_k(lib, M, N, 128)
        assert short_k(lib, M, N, 128, 2) and short_k(lib, M, N, 96) and short_k(lib, M, N + 8, 128)
    for M, N in ((2048, 2048), (8192, 1024), (4096, 2048), (511, 32768), (2048, 65536), (512, 20352)):
        assert short_k(lib, M, N, 128)


def test_few_rows_of_any_number_of_columns_stay_on_the_small_tiles(lib):
    for N in (129, 1000, 1001, 20001, 32767):
        assert not short_k(lib, 1, N, 128) and not short_k(lib, 8, N, 128)
        assert short_k(lib, 9, N, 128) and short_k(lib, 8, N, 64) and short_k(lib, 8, N, 96)
    assert short_k(lib, 1, 32769, 128) and short_k(lib, 1, 1000, 128, 33) and not short_k(lib, 1, 1000, 128, 32)     # 256 workgroups
    assert short_k(lib, 1, 40, 128) and short_k(lib, 1, 127, 96)
    assert not short_k(lib, 32, 1, 32) and not short_k(lib, 1, 15, 96) and short_k(lib, 33, 1, 32) and short_k(lib, 32, 8, 32)


def test_runs_of_tiles_that_change_column_stay_on_256_row_tiles(lib):
    for M in (129, 160, 192):
        for N in (21888, 28672, 32768):
            assert not short_k(lib, M, N, 128) and short_k(lib, M, N, 128, 2) and short_k(lib, M, N, 96)
        assert short_k(lib, M, 21760, 128) and short_k(lib, M, 32896, 128) and short_k(lib, M, 28680, 128)
    assert short_k(lib, 128, 28672, 128) and short_k(lib, 193, 28672, 128)


def scaled_plan(lib, M, N, K, may_split=True, cus=256):
    lib.mase_bench_scaled_plan.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int] * 2 + [ctypes.c_void_p]
    plan = (ctypes.c_int * 3)()
    assert lib.mase_bench_scaled_plan(M, N, K, cus, may_split, plan) == 0
    return tuple(plan)


def test_the_tile_plan_covers_k(lib):
    """Every share of a K split has macro steps, the last as well; the 256 x 256 kernel's are equal and even; no more workgroups than CUs."""
    for M in (65, 128, 200, 256, 300, 511, 1024, 3000, 16384):
        for N in (8, 264, 1000, 1024, 4096, 4104, 14336, 65536):
            for K in (512, 768, 1024, 2304, 4096, 4352, 14336, 14080):
                for cus in (256, 304, 64):
                    bn, splits, steps = scaled_plan(lib, M, N, K, True, cus)
                    nmac = K // 128
                    assert bn in (64, 128, 256) and 1 <= splits <= 16
                    assert (splits - 1) * steps < nmac <= splits * steps
                    assert splits == 1 or (steps >= 4 and splits * -(-M // (256 if bn == 256 else 128)) * -(-N // bn) <= cus)
                    assert bn != 256 or (splits * steps == nmac and steps % 2 == 0)
                    assert scaled_plan(lib, M, N, K, False, cus)[1:] == (1, nmac)


def test_few_tiles_of_a_long_k_share_it(lib):
    """The shapes on which the GPU tests compare a product in shares of K with the whole one."""
    for shape, plan in (((256, 256, 4096), (64, 8)), ((300, 520, 4096), (64, 4)), ((1024, 512, 14336), (128, 8)), ((700, 264, 7168), (64, 8))):
        assert scaled_plan(lib, *shape)[:2] == plan, shape
    assert scaled_plan(lib, 300, 520, 2048)[:2] == (64, 1)


def test_one_full_round_of_large_tiles_is_not_given_to_two_of_small_ones(lib):
    for M in (65, 96, 128):
        for K in (512, 1024, 2048):
            assert scaled_plan(lib, M, 65536, K) == (256, 1, K // 128)
    # one round of small tiles, a second that large ones would need as well, and several rows of tiles that share W
    for shape, bn in (((65, 28672, 4096), 128), ((128, 28672, 1024), 128), ((128, 98304, 4096), 128), ((128, 152064, 4096), 128), ((384, 14336, 512), 128),
                      ((200, 14336, 4096), 128), ((128, 14336, 4096), 64)):
        assert scaled_plan(lib, *shape)[0] == bn


def test_short_rows_behind_an_outer_axis_do_not_go_two_columns_to_a_lane(lib):
    """(matrices, rows, columns): a tenth to half slower than the other kernels there."""
    rule = lib.mase_bench_strided_pair_tiles
    rule.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int]

    def pair(outer, k, inner, bf16):
        return bool(rule(inner, outer * inner, k // 32, bf16))

    for shape in ((1000, 2080, 2), (32, 87360, 6), (1000, 672, 6), (128, 10912, 12), (8, 26208, 20), (11, 27776, 12), (1, 36832, 64), (29, 102272, 4), (128, 3584, 40)):
        assert not pair(*shape, 1), shape
    for shape in ((29, 69888, 4), (32, 131072, 4), (1000, 1024, 4), (1000, 352, 12), (64, 512, 64), (32, 1024, 64)):
        assert not pair(*shape, 0), shape
    for shape in ((1, 2976, 4096), (1, 65536, 200), (1, 1024, 2050), (4, 4096, 320), (1, 32768, 2), (8, 4096, 8), (3, 4096, 12)):
        assert pair(*shape, 1), shape
    for shape in ((1, 2976, 4096), (1, 65536, 200), (1, 1024, 2050), (128, 16384, 2), (32, 87360, 6), (32, 65536, 8), (64, 2048, 64)):
        assert pair(*shape, 0), shape


def test_ways_of_a_product_of_short_contraction():
    """2: queries and keys quantised inside the kernel of whole rows, 1: keys in a pass before it, 0: the general kernels."""
    from mase_hip.mxfp.kernels import scores_plan as plan

    for K in (32, 64, 96, 128):                     # few outputs: inside, whatever the shape
        assert plan(1, 8, K, 1, True) == plan(4096, 64, K, 17, True) == plan(1, 65536, K, 64, True) == plan(2000, 2000, K, 1, True) == 2
    assert plan(1536, 2048, 64, 8, True) == 2 and plan(1537, 2048, 64, 8, True) == 1      # twelve panels
    assert plan(512, 1000, 128, 48, True) == 2 and plan(513, 1000, 128, 48, True) == 1    # four
    # K = 96: zeros up to 128 and no prefetch
    assert plan(129, 8192, 96, 28, True) == plan(513, 2048, 96, 46, True) == plan(640, 8192, 96, 10, True) == plan(1000, 1000, 96, 10, True) == 0
    assert plan(128, 2048, 96, 127, True) == 2 and plan(16, 200, 96, 2507, True) == 0
    assert plan(1000, 1000, 96, 50, True) == plan(2048, 512, 96, 46, True) == 1
    # K = 128: long rows of whole lines, three to twelve panels
    assert plan(257, 2048, 128, 20, True) == plan(768, 65536, 128, 1, True) == plan(1464, 8192, 128, 5, True) == 0
    assert plan(256, 2048, 128, 20, True) == 2 and plan(768, 2040, 128, 31, True) == plan(768, 1984, 128, 31, True) == plan(2048, 2048, 128, 13, True) == 1
    # a dense A, or two formats: never inside
    for K in (32, 64, 96, 128):
        assert plan(1, 1000, K, 8, False) == plan(1000, 1000, K, 48, False) == plan(256, 512, K, 4, False) == 1
        assert plan(1, 1000, K, 400, False) == plan(2048, 2048, K, 32, False) == plan(513, 2048, K, 10, False) == plan(256, 1000, K, 200, False) == 0
    # what the kernel does not take, and empty products
    assert plan(64, 60, 64, 1, True) == plan(64, 64, 160, 1, True) == plan(64, 64, 48, 1, True) == plan(0, 64, 64, 1, True) == plan(64, 64, 64, 0, True) == 0
    assert plan(64, (1 << 23) + 8, 64, 1, True) == 0 and plan(2 ** 31 - 1, 8, 32, 1, True) == 0


def test_ragged_products_of_a_short_contraction_bring_no_room():
    """Their second launch would cost a call from Python more than sharing K saves on the GPU (the library splits them for who brings the room)."""
    from mase_hip.mxfp import kernels

    class Library:
        mase_hip_mxfp_gemm_workspace_bytes = staticmethod(lambda dense, M, N, K: 4096)

    def room(M, N, K):
        return kernels._workspace_bytes(Library, "no device", True, M, N, K)

    try:
        for M, N, K in ((1, 1000, 512), (16, 4001, 1312), (64, 1024, 1280), (65, 300, 992), (1000, 1673, 800), (200, 1024, 992), (129, 40, 896)):
            assert room(M, N, K) == 0, (M, N, K)
        for M, N, K in ((1, 1000, 1344), (64, 40, 4096), (65, 300, 1024), (1000, 1673, 2048), (65, 1024, 768), (512, 256, 512)):
            assert room(M, N, K) == 4096, (M, N, K)
    finally:
        for key in [k for k in kernels._WS_BYTES if k[0] == "no device"]:
            del kernels._WS_BYTES[key]


def test_few_rows_stay_with_the_weight_streaming_kernel_where_it_is_ahead(lib):
    """K of 1280 to 3584: tiles of 64 x 64 took 1.06 - 1.19 times as long for these (operand of x and product, another W on every call)."""
    for shape in ((1, 8192, 2048), (16, 8192, 2048), (1, 24576, 1536), (16, 20480, 1280), (5, 93008, 1792), (16, 48848, 2048), (1, 1536, 1280), (10, 1096, 1280),
                  (17, 8192, 2560), (32, 32768, 2560), (26, 4424, 2560), (17, 16384, 3072), (64, 4096, 3584), (64, 65536, 3072)):
        assert scaled_plan(lib, *shape)[0] == 0, shape
    for shape in ((1, 12288, 1024), (16, 14336, 768), (17, 65536, 512), (32, 8192, 1536), (33, 8192, 2048), (64, 8192, 2048), (48, 4096, 14336), (64, 14336, 4096)):
        assert scaled_plan(lib, *shape)[0] == 64, shape


def test_large_products_of_any_shape_stay_on_the_large_tiles(lib):
    """(batches, rows, columns, k) on both sides of the line; the first is the batch of odd products of the GPU tests."""
    rule = lib.mase_bench_any_shape
    rule.argtypes = [ctypes.c_int64] * 4 + [ctypes.c_int]
    for b, M, N, K in ((2, 4033, 2005, 2368), (1, 2759, 2961, 3648), (1, 16384, 14330, 4096)):
        assert not rule(M, N, K, b, 256), (b, M, N, K)
    for b, M, N, K in ((2, 1001, 1003, 2368), (1, 4033, 2005, 160), (40, 257, 259, 96), (1, 700, 1000, 4096)):
        assert rule(M, N, K, b, 256), (b, M, N, K)
