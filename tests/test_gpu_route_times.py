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
