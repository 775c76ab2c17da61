"""Extract down the rows of 16-bit matrices with an even inner axis, two columns to a lane: columns and k-blocks that fill tiles of 128 x 4
and that do not, several outer matrices in one tile, every fp16 and bf16 bit pattern as an element and as the largest of its block, inf
and NaN blocks beside ordinary ones; codes and scales against the checker bit for bit."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


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
