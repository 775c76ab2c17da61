"""The short-contraction GEMM kernel (K <= 128, no bias) at the edges of its tiles: rows around the 64-row A tile, columns around the
128-column W tile, rows of y that are and are not multiples of 16 bytes and of whole lines, contractions that fill the 64- or 128-k
loops or leave zero-filled k behind, one tile and several per workgroup (with the counted wait between tiles of one column, and
across columns and products), products sharing an operand, block scales on the slow compose route.  The compose itself, every
scale and code, is pinned in test_gpu_gemm_compose_exact.py."""
import pytest
import torch

import oracle
from helpers import PRESETS

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
TAGS = list(PRESETS)


@pytest.mark.parametrize("odt", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("K", [32, 64, 96, 128])
@pytest.mark.parametrize("M,N", [(1, 8), (63, 127), (64, 128), (65, 129), (33, 64), (33, 72), (64, 136), (9, 1001), (200, 1000), (130, 1), (700, 72)])
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


def _bound(a, w, ref, odt):
    """fp32 sums of at most 128 products of exact operands: 128 * 2^-24 of the sum of magnitudes, then the rounding to the output type."""
    rounding = {torch.float32: 2.0 ** -24, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[odt]
    return 128 * 2.0 ** -24 * torch.matmul(a.abs(), w.abs().transpose(-1, -2)) + rounding * ref.abs() + (2.0 ** -24 if odt == torch.float16 else 0.0)


# tiles = batches * ceil(M / 64) * ceil(N / 128): more than the 512 workgroups of a 256-CU device, so that workgroups take a second tile
# of the same column while the first one's stores are in flight, and go on to other columns and products
@pytest.mark.parametrize("odt", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("B,M,N,K", [
    (9, 1000, 1000, 128),     # 1152 tiles; 2000- or 4000-byte rows: 16-byte stores, rows that are no whole lines; 40 rows in the last tile
    (5, 1100, 1024, 96),      # 720 tiles; whole-line rows, zero-filled k
    (1, 5000, 1001, 128),     # 632 tiles; odd rows: element stores, no counted wait
    (2, 3000, 840, 64),       # 658 tiles on the 64-k loops
    (40, 129, 520, 32),       # 600 tiles, three per column: most runs cross columns, some products
])
def test_short_k_several_tiles_per_workgroup(B, M, N, K, odt):
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(M + N + K)
    for tag in ("MXFP8_E4M3_fn", "OCP_MXFP4_E2M1"):
        e, m = PRESETS[tag]
        meta = MXFPMeta(32, 8, e, m, True, "rn")
        a = torch.randn(B, M, K, generator=g).to(torch.bfloat16)
        w_el = torch.randint(0, 1 << (1 + e + m), (B * N * K // 32, 32), generator=g, dtype=torch.uint8)
        w_sc = torch.randint(110, 122, (B * N * K // 32, 1), generator=g, dtype=torch.uint8)
        w = oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.float32).view(B, N, K).double()
        if B == 1:
            y = mxk.mxfp_gemm(a[0].to(DEV), None, None, None, w_sc.to(DEV), w_el.to(DEV), meta, None, M, N, K, odt)[None]
        else:
            y = mxk.mxfp_gemm_batched(a.to(DEV).reshape(-1), w_sc.to(DEV), w_el.to(DEV), meta, B, M, N, K, odt, M * K, N * K)
        ref = torch.matmul(a.double(), w.transpose(1, 2))
        d = (y.cpu().double() - ref).abs()
        assert bool((d <= _bound(a.double(), w, ref, odt)).all()), (tag, float(d.max()))


def test_short_k_scales_on_the_slow_route():
    """Blocks whose scale byte the hardware convert does not take beside ordinary ones in the same wavefront, every format.  Each row of A
    selects one k, so every output is one value of W.  A third of the blocks have scales 244 .. 254, with the codes that would leave
    bf16's range replaced by zeros: the outputs are exact.  Every 40th row of W holds a block of scale 255 (all inf and NaN): its column
    is NaN and no other."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFPMeta

    g = torch.Generator().manual_seed(5)
    M, N, K = 70, 200, 128
    for tag in TAGS:
        e, m = PRESETS[tag]
        k_of = torch.randint(0, K, (M,), generator=g)
        w_el = torch.randint(0, 1 << (1 + e + m), (N * K // 32, 32), generator=g, dtype=torch.uint8)
        w_sc = torch.randint(20, 244, (N * K // 32, 1), generator=g, dtype=torch.uint8)
        w_sc[::3] = torch.randint(244, 255, w_sc[::3].shape, generator=g, dtype=torch.uint8)
        w_el[~oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.bfloat16).view(-1, 32).isfinite()] = 0
        bad = torch.arange(N) % 40 == 7
        w_sc.view(N, K // 32)[bad, 2] = 255
        w = oracle.compose_mxfp(w_sc, w_el, 32, e, m, True, torch.bfloat16).view(N, K)
        assert w[~bad].isfinite().all() and (w[~bad].float()[:, k_of] != 0).double().mean() > 0.5
        for scale in (1.0, 2.0 ** -100):
            a = torch.zeros(M, K)
            a[torch.arange(M), k_of] = scale
            y = mxk.mxfp_gemm(a.to(torch.bfloat16).to(DEV), None, None, None, w_sc.to(DEV), w_el.to(DEV), MXFPMeta(32, 8, e, m, True, "rn"), None, M, N, K,
                              torch.float32).cpu()
            want = (w.double()[:, k_of].T * scale)[:, ~bad]
            got = y[:, ~bad]
            assert y[:, bad].isnan().all() and not got.isnan().any(), tag
            normal = (want.abs() >= 2.0 ** -126) | (want == 0)
            assert torch.equal(got.double()[normal], want[normal]), (tag, scale)
            assert bool((got.abs()[~normal] < 2.0 ** -126).all()), (tag, scale)      # subnormal products: kept or flushed by the matrix unit
            assert normal.double().mean() > 0.5, (tag, scale)


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


def test_transposed_right_operand_on_the_block_scaled_route():
    """The same where the product takes the block-scaled GEMM (one matrix, 512 rows or more, K a multiple of 256): both layouts of the
    right operand, with and without unit batch axes, bit for bit, and against the oracle's quantisation."""
    import mase_hip.mxfp.functional as F
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    g = torch.Generator().manual_seed(8)
    k = (0.1 * torch.randn(264, 768, generator=g)).to(torch.bfloat16)
    q = torch.randn(2, 300, 768, generator=g).to(torch.bfloat16)
    calls = []
    real = mxk.mxfp_gemm_scaled
    mxk.mxfp_gemm_scaled = lambda *a, **kw: (calls.append(1), real(*a, **kw))[1]
    try:
        y = F.mxfp_matmul(q.to(DEV), k.to(DEV).transpose(-1, -2), fmt, fmt, "XqWq", "fused")
        for other in (k.to(DEV).transpose(-1, -2).contiguous(), k.to(DEV)[None].transpose(-1, -2)):
            y2 = F.mxfp_matmul(q.to(DEV), other, fmt, fmt, "XqWq", "fused")
            assert y2.shape == y.shape and torch.equal(y.view(torch.int16), y2.view(torch.int16))
    finally:
        mxk.mxfp_gemm_scaled = real
    assert len(calls) == 3, "not the route this test is for"
    ref = torch.matmul(oracle.qdq_mxfp(q, 32, 4, 3).double(), oracle.qdq_mxfp(k, 32, 4, 3).double().T).to(torch.bfloat16).double()
    assert ((y.cpu().double() - ref).norm() / ref.norm()).item() <= 1e-3
