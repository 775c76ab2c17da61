"""The short-contraction GEMM kernel (K <= 128, no bias) at the edges of its tiles: rows around the 64-row A tile, columns around the
128-column W tile, rows of y that are and are not multiples of 16 bytes, contractions that fill the 64- or 128-k loops or leave
zero-filled k behind, one tile and many per workgroup, products sharing an operand, block scales on the slow compose route."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TAGS = list(PRESETS)


@pytest.mark.parametrize("odt", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
@pytest.mark.parametrize("M,N", [(1, 8), (63, 127), (64, 128), (65, 129), (33, 64), (200, 1000), (130, 1), (700, 72)])
def test_short_k_against_float64(M, N, K, odt):
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(M * 1000 + N + K)
    for i, tag in enumerate(TAGS):
        e, m = PRESETS[tag]
        a = torch.randn(M, K, generator=g).to(torch.bfloat16)
        w_el = torch.randint(0, 1 << (1 + e + m), (N * K // 32, 32), generator=g, dtype=torch.uint8)
        w_sc = torch.randint(110, 131, (N * K // 32, 1), generator=g, dtype=torch.uint8)
        w = oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.float32).view(N, K)
        y = mxk.mxfp_gemm(a.to(DEV), None, None, None, w_sc.to(DEV), w_el.to(DEV), MXFPMeta(32, 8, e, m, True, "rn"), None, M, N, K, odt)
        ref = a.double() @ w.double().T
        # fp32 sums of at most 128 products of exact operands: 128 * 2^-24 of the sum of magnitudes, then the rounding to the output type
        bound = 128 * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[odt] * ref.abs()
        if odt == torch.float16:
            bound += 2.0 ** -24
            ref = torch.where(ref.abs() < 65504, ref, torch.full_like(ref, float("nan")))   # out of range: not compared
        d = (y.cpu().double() - ref).abs()
        assert ((d <= bound) | ref.isnan()).all(), (tag, d.max())


def test_short_k_scales_on_the_slow_route():
    """Scale bytes that the hardware convert does not take (255: "times inf") beside ordinary ones, every format."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(5)
    M, N, K = 70, 200, 128
    for tag in TAGS:
        e, m = PRESETS[tag]
        a = torch.zeros(M, K)
        a[torch.arange(M), torch.randint(0, K, (M,), generator=g)] = 2.0 ** -100          # one element per row: y = one value of W, scaled
        w_el = torch.randint(0, 1 << (1 + e + m), (N * K // 32, 32), generator=g, dtype=torch.uint8)
        w_sc = torch.randint(0, 255, (N * K // 32, 1), generator=g, dtype=torch.uint8)
        w_sc[::3] = torch.randint(244, 256, (w_sc[::3].shape), generator=g, dtype=torch.uint8)
        w = oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.bfloat16).view(N, K)
        y = mxk.mxfp_gemm(a.to(torch.bfloat16).to(DEV), None, None, None, w_sc.to(DEV), w_el.to(DEV), MXFPMeta(32, 8, e, m, True, "rn"), None, M, N, K,
                          torch.float32).cpu()
        want = (a[:, None, :] * w.float()[None]).sum(-1)     # (inf and NaN anywhere in a row of W make the whole column NaN here and there)
        tiny = want.abs() < 2.0 ** -126                       # subnormal products: flushed by the matrix unit
        same = (y == want) | (y.isnan() & want.isnan()) | tiny
        assert same.all(), tag


def test_short_k_batches_and_shared_operands():
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    g = torch.Generator().manual_seed(9)
    for B, M, N, K in ((40, 96, 160, 64), (3, 1000, 1000, 128), (700, 8, 264, 32)):
        for a_shared, w_shared in ((False, False), (True, False), (False, True)):
            a = torch.randn((1 if a_shared else B), M, K, generator=g).to(torch.bfloat16)
            w_el = torch.randint(0, 256, ((1 if w_shared else B) * N * K,), generator=g, dtype=torch.uint8)
            w_sc = torch.randint(118, 126, (w_el.numel() // 32,), generator=g, dtype=torch.uint8)
            y = mxk.mxfp_gemm_batched(a.to(DEV).reshape(-1), w_sc.to(DEV), w_el.to(DEV), fmt, B, M, N, K, torch.bfloat16, 0 if a_shared else M * K,
                                      0 if w_shared else N * K)
            w = oracle.compose_mxfp(w_sc, w_el, 32, 4, 3, True, torch.float32).view(-1, N, K)
            ref = torch.matmul(a.float(), w.transpose(1, 2)).to(torch.bfloat16).double()
            err = ((y.cpu().double() - ref).norm() / ref.norm()).item()
            assert err <= 1e-3, (B, M, N, K, a_shared, w_shared, err)


@pytest.mark.parametrize("shape", [(2, 3, 100, 64), (5, 72, 128), (96, 256)])
def test_transposed_right_operand_is_quantised_where_it_lies(shape):
    """``other`` as the transposed view of a contiguous tensor (keys of an attention product): same bits as from a contiguous copy."""
    import mase_hip.mxfp.functional as F
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    g = torch.Generator().manual_seed(3)
    k = torch.randn(*shape, generator=g).to(torch.bfloat16).to(DEV)
    q = torch.randn(*shape[:-2], 40, shape[-1], generator=g).to(torch.bfloat16).to(DEV)
    for func_type in ("XqWq", "XWq"):
        y = F.mxfp_matmul(q, k.transpose(-1, -2), fmt, fmt, func_type, "fused")
        y2 = F.mxfp_matmul(q, k.transpose(-1, -2).contiguous(), fmt, fmt, func_type, "fused")
        assert torch.equal(y.view(torch.int16), y2.view(torch.int16))
