"""Calls whose kernel was once the wrong one for their size, held to a time: each against another call of this library that does the
same work by another route.  The margins lie between the two routes' measured times; GPU time only (graph replays, the best of several)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def gpu_us(f, calls=20):
    """Microseconds of one call of `f` on the GPU: `calls` of them in a graph, the best of seven replays."""
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        f()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        for _ in range(calls):
            f()
    best = float("inf")
    with torch.cuda.stream(stream):
        for _ in range(8):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record(stream)
            graph.replay()
            end.record(stream)
            end.synchronize()
            best = min(best, start.elapsed_time(end) * 1000 / calls)
    return best


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("columns", [65, 193])
def test_extract_down_the_rows_with_a_last_tile_of_few_columns(dt, columns):
    """One column in the last tile of 64 against seventeen: 9.0 against 4.1 us when its wavefronts ran with one lane of 64 enabled."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    few, more = (torch.randn(1024, c, device=DEV).to(dt) for c in (columns, columns + 16))
    t_few, t_more = (gpu_us(lambda x=x: mxk.extract_mxfp_components_strided(x, 0, fmt)) for x in (few, more))
    assert t_few <= 1.4 * t_more, (t_few, t_more)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, torch.bfloat16])
def test_extract_down_one_long_column(dt):
    """One column is the flat tensor: the kernels for blocks down the rows may cost a few times the flat one's time (7 against 3 us),
    not 15 times (one lane of a wavefront at work: 47 - 54 us)."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    x = torch.randn(1 << 20, 1, device=DEV).to(dt)
    t, t_flat = gpu_us(lambda: mxk.extract_mxfp_components_strided(x, 0, fmt)), gpu_us(lambda: mxk.extract_mxfp_components(x.view(-1), fmt))
    assert t <= 4 * t_flat, (t, t_flat)


def _product(M, N, K, batches=1):
    g = torch.Generator(device=DEV).manual_seed(M + N)
    a = torch.randn(batches * M, K, generator=g, device=DEV).to(torch.bfloat16)
    el = torch.randint(0, 256, (batches * N * K,), generator=g, device=DEV, dtype=torch.uint8)
    sc = torch.randint(118, 126, (batches * N * K // 32,), generator=g, device=DEV, dtype=torch.uint8)
    return a, sc, el


@pytest.mark.parametrize("M,N", [(1, 4096), (16, 14336), (32, 4096), (64, 1024), (64, 8192)])
def test_short_contraction_of_few_rows(M, N):
    """Without a bias the product may not take longer than with one, which always runs on the weight-streaming kernels here (0.83 - 0.92 of
    its time, 1.1 - 1.9 times as long on the kernel for short contractions)."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    a, sc, el = _product(M, N, 128)
    bias = torch.randn(N, device=DEV).to(torch.bfloat16)
    t, t_bias = (gpu_us(lambda b=b: mxk.mxfp_gemm(a, None, None, None, sc, el, fmt, b, M, N, 128, torch.bfloat16)) for b in (None, bias))
    assert t <= 1.05 * t_bias, (t, t_bias)


@pytest.mark.parametrize("M,N,odt", [(1024, 14336, torch.bfloat16), (512, 28672, torch.bfloat16), (3000, 4096, torch.bfloat16), (16384, 4096, torch.float32)])
def test_short_contraction_of_a_full_round_of_large_tiles(M, N, odt):
    """The same for one product of at least 160 tiles of 512 x 128: 10.7 us at 1024 x 14336 with a bias, 16.4 on the kernel for short
    contractions."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    a, sc, el = _product(M, N, 128)
    bias = torch.randn(N, device=DEV).to(torch.bfloat16)
    t, t_bias = (gpu_us(lambda b=b: mxk.mxfp_gemm(a, None, None, None, sc, el, fmt, b, M, N, 128, odt)) for b in (None, bias))
    assert t <= 1.2 * t_bias, (t, t_bias)


def test_attention_scores_of_one_query():
    """One query per head against 2048 keys of 8 heads: 4.8 us on the weight-streaming kernel, 6.4 on the kernel for short contractions.
    Held to the time of one product with as many rows of W and a bias (0.82 of it, 1.1 times)."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    B, M, N, K = 8, 1, 2048, 128
    a, sc, el = _product(M, N, K, B)
    bias = torch.randn(B * N, device=DEV).to(torch.bfloat16)
    t = gpu_us(lambda: mxk.mxfp_gemm_batched(a.view(-1), sc, el, fmt, B, M, N, K, torch.bfloat16, M * K, N * K))
    t_one = gpu_us(lambda: mxk.mxfp_gemm(a[:1], None, None, None, sc, el, fmt, bias, 1, B * N, K, torch.bfloat16))
    assert t <= t_one, (t, t_one)


@pytest.mark.parametrize("N,aligned", [(1001, 1000), (10010, 10008)])
def test_short_contraction_of_one_row_and_an_odd_number_of_columns(N, aligned):
    """Rows of y at no alignment leave element by element; only those there are (4.6 us when all 32 rows of a tile were stepped through,
    3.8 as with whole 16-byte stores).  Held to a multiple of 8 columns."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    t = []
    for n in (N, aligned):
        a, sc, el = _product(1, n, 64)
        t.append(gpu_us(lambda: mxk.mxfp_gemm(a, None, None, None, sc, el, fmt, None, 1, n, 64, torch.bfloat16)))
    assert t[0] <= 1.1 * t[1], t


@pytest.mark.parametrize("M,N,most", [(1, 20008, 1.05), (129, 28672, 0.9), (192, 24576, 0.85)])
def test_short_contractions_between_the_tile_sizes(M, N, most):
    """One row of a number of columns that the weight-streaming kernels do not take, and rows whose tiles leave runs that change column:
    held to the same product with a bias, on the kernels for long contractions (5.7, 8.8 and 9.2 us against 6.0, 11.5 and 12.7 with the
    bias; 6.6, 12.7 and 12.5 on the other)."""
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    a, sc, el = _product(M, N, 128)
    bias = torch.randn(N, device=DEV).to(torch.bfloat16)
    t, t_bias = (gpu_us(lambda b=b: mxk.mxfp_gemm(a, None, None, None, sc, el, fmt, b, M, N, 128, torch.bfloat16)) for b in (None, bias))
    assert t <= most * t_bias, (t, t_bias)


@pytest.mark.parametrize("B,M,N,K,quantised", [(46, 513, 2048, 96, True), (10, 640, 8192, 96, True), (12, 384, 2048, 96, True), (6, 768, 2048, 128, True), (1, 768, 65536, 128, True),
                                               (360, 1, 512, 64, False)])
def test_attention_scores_against_the_general_kernels(B, M, N, K, quantised):
    """Shapes for which a pass over each operand and the kernels that compose codes are ahead of the kernel that quantises on the way in
    (1.27 - 1.55 times as long there; the same kernels through the two calls come out up to 1.09 apart)."""
    import mase_hip.mxfp.functional as MX
    import mase_hip.mxfp.kernels as mxk
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn as fmt

    q, k = (torch.randn(B, n, K, device=DEV).to(torch.bfloat16) for n in (M, N))

    def general():
        a = mxk.quantize_dequantize(q.view(-1), fmt, torch.bfloat16) if quantised else q.view(-1)
        sc, el = mxk.extract_mxfp_components(k.view(-1), fmt)
        return mxk.mxfp_gemm_batched(a, sc.view(-1), el.view(-1), fmt, B, M, N, K, torch.bfloat16, M * K, N * K)

    t = gpu_us(lambda: MX.mxfp_matmul(q, k.transpose(-1, -2), fmt, fmt, "XqWq" if quantised else "XWq", "fused"), 8)
    t_general = gpu_us(general, 8)
    assert t <= 1.15 * t_general, (t, t_general)
