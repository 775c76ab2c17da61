"""Extract down the rows of 16-bit matrices with an even inner axis, codes and scales against the checker bit for bit: sizes on both sides
of the rule that takes them two columns to a lane, and, on that kernel by the rule's own answer, columns and k-blocks that fill tiles of
128 x 4 and that do not, several outer matrices in one tile, every fp16 and bf16 bit pattern as an element and as the largest of its block, inf
and NaN blocks beside ordinary ones."""
import ctypes
import os

import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _two_columns_to_a_lane(shape, dim, dtype):
    """Is mxfp_strided_pair_kernel what an extract of such a tensor runs?"""
    lib = ctypes.CDLL(os.path.join(ROOT, "mase-triton_amd", "mase_hip", "lib", "libmase_bench.so"))
    lib.mase_bench_strided_pair_tiles.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_int]
    k, inner, columns = shape[dim], 1, 1
    for i, d in enumerate(shape):
        inner *= d if i > dim else 1
        columns *= d if i != dim else 1
    bf16 = dtype == torch.bfloat16
    whole_lines = bf16 and inner % 128 == 0 and k % 128 == 0           # a kernel of their own
    return inner % 2 == 0 and not whole_lines and bool(lib.mase_bench_strided_pair_tiles(inner, columns, k // 32, bf16))


def _check(x, block_dim, tag):
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.meta as meta

    sc, el, _ = MX.extract_mxfp_components(x.to(DEV), block_dim, getattr(meta, tag))
    rot = x.movedim(block_dim, -1).contiguous().view(-1)
    rs, re = oracle.extract_mxfp(rot, 32, *PRESETS[tag])
    assert torch.equal(sc.cpu().view(-1), rs.view(-1)) and torch.equal(el.cpu().view(-1), re.view(-1))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,dim", [((32, 2), 0), ((96, 126), 0), ((128, 128), 0), ((160, 130), 0), ((2048, 258), 0), ((256, 9000), 0), ((4128, 512), 0), ((32, 65538), 0),
                                       ((5, 64, 50), 1), ((3, 224, 4, 46), 1), ((700, 128, 6), 1), ((40, 1024, 8), 1)])
def test_pairs_of_columns(dtype, shape, dim):
    g = torch.Generator().manual_seed(sum(shape))
    x = torch.randn(*shape, generator=g) * torch.exp(4 * torch.randn(*shape[:-1], 1, generator=g))
    for tag in PRESETS:
        _check(x.to(dtype), dim, tag)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tag", list(PRESETS))
def test_every_pattern(dtype, tag):
    """Column c of the first matrix holds 32 neighbouring bit patterns (each its block's neighbourhood); in the others every pattern lies below
    a block maximum of each binade that the pattern does not exceed, beside one of inf and NaN."""
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    _check(bits.view(2048, 32).t().contiguous().view(dtype).repeat(2, 1).contiguous(), 0, tag)       # 64 rows, every pattern twice
    g = torch.Generator().manual_seed(7)
    x = bits[torch.randperm(65536, generator=g)].view(128, 512).repeat(8, 1).view(dtype).clone()       # inf / NaN in most wavefronts
    _check(x, 0, tag)
    finite = bits[bits.view(dtype).isfinite()]
    n = finite.numel() // 512 * 512
    for top in ([-14, -2, 3, 15] if dtype == torch.float16 else [-100, -14, 0, 20, 127]):
        x = finite[torch.randperm(finite.numel(), generator=g)[:n]].view(-1, 512)
        x = x[:x.shape[0] // 32 * 32].clone().view(dtype)
        x = torch.where(x.abs().double() < 2.0 ** top, x, torch.zeros_like(x))
        x.view(-1, 32, 512)[:, 5] = torch.tensor(2.0 ** top * 1.5, dtype=torch.float64).to(dtype)
        _check(x, 0, tag)
        _check(x.repeat(4, 1), 0, tag)


PAIR_SHAPES = [(s, d, t) for t in (torch.float16, torch.bfloat16) for s, d in
               (((1024, 2050), 0), ((1056, 2048), 0), ((1056, 2050), 0), ((992, 2174), 0), ((3, 1056, 700), 1), ((6, 352, 1030), 1), ((2, 1088, 5, 206), 1))]
PAIR_SHAPES += [((350, 1056, 6), 1, torch.float16), ((8, 1056, 6), 1, torch.bfloat16), ((3, 2080, 20), 1, torch.bfloat16), ((1056, 2), 0, torch.bfloat16)]


@pytest.mark.parametrize("shape,dim,dtype", PAIR_SHAPES)
def test_two_columns_to_a_lane(dtype, shape, dim):
    """Last tiles of 2 to 126 columns and of one to three k-blocks, outer matrices that end inside a tile; inf and NaN in some blocks."""
    assert _two_columns_to_a_lane(shape, dim, dtype)
    g = torch.Generator().manual_seed(sum(shape))
    x = (torch.randn(*shape, generator=g) * torch.exp(3 * torch.randn(*shape[:-1], 1, generator=g))).to(dtype)
    flat = x.view(-1)
    for i, v in enumerate((float("inf"), float("-inf"), float("nan"))):
        flat[torch.randint(0, flat.numel(), (200,), generator=g)] = v
        flat[-1 - 5 * i] = v
    for tag in PRESETS:
        _check(x, dim, tag)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("tag", list(PRESETS))
def test_every_pattern_two_columns_to_a_lane(dtype, tag):
    """1056 x 2050 on that kernel: every bit pattern among its neighbours; every one in random company (fp16: inf or NaN in two blocks of
    three); every finite one below block maxima of several binades."""
    rows, columns = 1056, 2050
    assert _two_columns_to_a_lane((rows, columns), 0, dtype)
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    g = torch.Generator().manual_seed(11)
    near = torch.cat([bits.view(2048, 32).t(), bits[:64].view(32, 2)], 1)                 # 32 neighbours to a column
    _check(torch.cat([near.roll(i, 1) for i in range(rows // 32)]).view(dtype).contiguous(), 0, tag)

    def mixed(patterns):
        n = -(-rows * columns // patterns.numel())
        return torch.cat([patterns[torch.randperm(patterns.numel(), generator=g)] for _ in range(n)])[:rows * columns].view(rows, columns).contiguous()

    _check(mixed(bits).view(dtype), 0, tag)
    finite = bits[bits.view(dtype).isfinite()]
    for top in ([-14, -2, 3, 15] if dtype == torch.float16 else [-100, -14, 0, 20, 127]):
        x = mixed(finite).view(dtype)
        x = torch.where(x.abs().double() < 2.0 ** top, x, torch.zeros_like(x))
        x.view(-1, 32, columns)[:, 5] = torch.tensor(2.0 ** top * 1.5, dtype=torch.float64).to(dtype)
        _check(x, 0, tag)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tag", list(PRESETS))
def test_nonfinite_blocks_one_column_to_a_lane(dtype, tag):
    """An odd number of columns: blocks of inf and of NaN with every payload beside ordinary blocks, zeros and blocks for the general routine
    (scales below the format's bias or past 150) in one wavefront."""
    g = torch.Generator().manual_seed(13)
    rows, columns = 128, 513
    if dtype == torch.float32:
        x = torch.randn(rows, columns, generator=g)
        bits = x.view(torch.int32).view(-1)
        some = torch.randperm(rows * columns, generator=g)[:3000]
        bits[some] = 0x7F800000 | (torch.randint(0, 1 << 23, (3000,), generator=g).to(torch.int32) << torch.randint(0, 23, (3000,), generator=g).to(torch.int32) & 0x7FFFFF)
        bits[some[::2]] |= -(1 << 31)
    else:
        x = torch.arange(65536, dtype=torch.int32).to(torch.int16)[torch.randperm(65536, generator=g)].view(dtype)
        x = torch.cat([x, x[:rows * columns - 65536]]).view(rows, columns).contiguous()
    _check(x, 0, tag)
    sparse = torch.randn(rows, columns, generator=g).to(dtype)
    sparse[:, ::7] = 0.0
    if dtype != torch.float16:
        sparse[:, 3::11] *= 1e30
        sparse[:, 4::13] *= 1e-37
    sparse[5, ::5], sparse[77, 1::9], sparse[100, 2::17] = float("inf"), float("nan"), float("-inf")
    _check(sparse, 0, tag)
