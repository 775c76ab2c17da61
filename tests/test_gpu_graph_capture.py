"""The library enqueues kernels only (no allocation, no synchronisation, no memset), so a quantised layer can be
captured into a HIP graph and replayed: decode-size calls are launch-bound otherwise.  Every replay is checked
against the eager result, with eager work and synchronisations between the replays."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("M,K,N", [(8, 512, 12288), (200, 512, 12288), (1024, 512, 12288),
                                   (200, 4096, 512),    # K split over workgroups, workspace from torch's allocator
                                   (16, 4096, 1024), (40, 4096, 1024),   # the weight-streaming kernel: one and three operand tiles of x
                                   (48, 8192, 520)])    # ... on K slices: workspace and the reduce kernel inside the capture
def test_fused_layer_replays_from_a_graph(M, K, N):
    from mase_hip import _lib
    from mase_hip.mxfp.layers import MXFPLinearPTQ
    from mase_hip.mxfp.meta import MXFP8_E4M3_fn, OCP_MXFP6_E3M2

    _lib.load()
    lin = torch.nn.Linear(K, N, bias=True, dtype=torch.bfloat16, device=DEV)
    layer = MXFPLinearPTQ.from_linear(lin, MXFP8_E4M3_fn, OCP_MXFP6_E3M2, None, "XqWqB", "fused")
    g = torch.Generator(device=DEV).manual_seed(M)
    static_x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # warm-up outside the capture: first-call set-up of the kernels happens here
        for _ in range(3):
            layer(static_x)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_y = layer(static_x)
    for i in range(4):
        x = torch.randn(M, K, generator=g, device=DEV).to(torch.bfloat16) * (i + 1)
        want = layer(x)                     # eager work between the replays
        torch.cuda.synchronize()
        static_x.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(static_y.view(torch.int16), want.view(torch.int16)), f"replay {i}"


@pytest.mark.parametrize("family", ["mxfp", "minifloat"])
@pytest.mark.parametrize("layer_type,rows,warm_rows", [("XqWqB", 48, 2000),   # the packed weight's rows, warmed up at the block-scaled form's
                                                       ("XWqB", 12, 40),      # weight only: warmed up on the components
                                                       ("XWqB", 3000, 12),    # ... and the bf16 kernel's prepared form
                                                       ("XqWqB", 48, None)])  # no warm-up but of another layer
def test_forms_that_a_capture_meets_first(family, layer_type, rows, warm_rows):
    """A layer captured at a row count whose form of the weight it has not built: eager calls before the first replay, and of other streams, are right, and
    so is every replay."""
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.meta as mx
    from mase_hip.minifloat.layers import MinifloatLinearPTQ
    from mase_hip.mxfp.layers import MXFPLinearPTQ

    K, N = 4096, 2048
    g = torch.Generator(device=DEV).manual_seed(rows)
    w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)

    def make(backend):
        if family == "mxfp":
            return MXFPLinearPTQ(w, None, mx.MXFP8_E4M3_fn if layer_type == "XqWqB" else None, mx.OCP_MXFP4_E2M1, None, layer_type, backend)
        return MinifloatLinearPTQ(weight=w, bias=None, x_minifloat_meta=mf.FP8_E4M3_fn if layer_type == "XqWqB" else None, w_minifloat_meta=mf.FP4_E2M1_fn,
                                  b_minifloat_meta=None, layer_type=layer_type, backend=backend)

    def close(y, ref):
        return ((y.double() - ref.double()).norm() / ref.double().norm()).item() <= 1e-3

    layer, separate, other = make("fused"), make("separate"), make("fused")
    x = torch.randn(rows, K, generator=g, device=DEV).to(torch.bfloat16)
    want = separate(x)
    if warm_rows is not None:
        layer(torch.randn(warm_rows, K, generator=g, device=DEV).to(torch.bfloat16))
    other(x)                                       # the kernels' first launches are not captured
    torch.cuda.synchronize()
    static_x, graph = x.clone(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        static_y = layer(static_x)
    assert close(layer(x), want) and close(layer(x), want)
    for i in range(3):
        scale = 2.0 ** i
        static_x.copy_(x * scale)
        graph.replay()
        torch.cuda.synchronize()
        assert close(static_y, separate(x * scale)), i
        assert close(layer(x), want), i
    assert close(other(x), want)


@pytest.mark.parametrize("family", ["mxfp", "minifloat"])
@pytest.mark.parametrize("layer_type,rows", [("XqWqB", 48), ("XqWqB", 2000), ("XWqB", 12), ("XWqB", 3000), ("XWqB", 100)])
def test_replays_follow_a_weight_that_is_loaded_in_place(family, layer_type, rows):
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.meta as mx
    from mase_hip.minifloat.layers import MinifloatLinearPTQ
    from mase_hip.mxfp.layers import MXFPLinearPTQ

    K, N = 4096, 2048
    g = torch.Generator(device=DEV).manual_seed(rows)

    def make():
        w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
        if family == "mxfp":
            return MXFPLinearPTQ(w, None, mx.MXFP8_E4M3_fn if layer_type == "XqWqB" else None, mx.OCP_MXFP4_E2M1, None, layer_type, "fused")
        return MinifloatLinearPTQ(weight=w, bias=None, x_minifloat_meta=mf.FP8_E4M3_fn if layer_type == "XqWqB" else None, w_minifloat_meta=mf.FP4_E2M1_fn,
                                  b_minifloat_meta=None, layer_type=layer_type, backend="fused")

    layers = [make() for _ in range(3)]
    x = torch.randn(rows, K, generator=g, device=DEV).to(torch.bfloat16)
    want = [layer(x) for layer in layers]
    torch.cuda.synchronize()
    layer, graph = layers[0], torch.cuda.CUDAGraph()
    states = [{k: v.clone() for k, v in other.state_dict().items()} for other in layers]
    with torch.cuda.graph(graph):
        y = layer(x)
    for i in (0, 1, 2, 1, 0):
        layer.load_state_dict(states[i])
        if i == 2:
            assert torch.equal(layer(x), want[i])
        junk = [torch.full((N * K,), 255, dtype=torch.uint8, device=DEV) for _ in range(4)]      # what memory that was given back would hold now
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want[i]), i
        del junk
    with torch.no_grad():                                       # a write in place, seen with the next call
        for name, p in layer.named_parameters():
            p.copy_(states[1][name])
    assert torch.equal(layer(x), want[1])
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(y, want[1])


def test_one_call_before_the_capture_is_enough():
    """The capture finds a form that no other call has asked about since: the query does not end the capture, and the form is read, not built again."""
    import mase_hip.mxfp.meta as mx
    from mase_hip import _lib
    from mase_hip.mxfp.layers import MXFPLinearPTQ

    g = torch.Generator(device=DEV).manual_seed(1)
    w = torch.randn(2048, 4096, generator=g, device=DEV).to(torch.bfloat16)
    x = torch.randn(12, 4096, generator=g, device=DEV).to(torch.bfloat16)
    layer = MXFPLinearPTQ(w, None, None, mx.OCP_MXFP4_E2M1, None, "XWqB", "fused")
    want = layer(x)
    torch.cuda.synchronize()
    form, graph = layer._packed_w, torch.cuda.CUDAGraph()
    assert form.stream is not None
    with torch.cuda.graph(graph):
        y = layer(x)
    assert layer._packed_w is form and form.stream is None
    side, busy = torch.cuda.Stream(), torch.randn(4096, 4096, device=DEV)
    torch.cuda.synchronize()
    with torch.cuda.stream(side):                  # an event that is still to come
        for _ in range(20):
            torch.mm(busy, busy)
        event = side.record_event()
    early = _lib.stream_done(side, event), _lib.stream_done(side)
    side.synchronize()
    assert early == (False, False) and _lib.stream_done(side, event) and _lib.stream_done(side)
    again = torch.cuda.CUDAGraph()
    with torch.cuda.graph(again, stream=side):     # a stream that is captured has not run what it was given
        x.add_(0)
        assert not _lib.stream_done(side) and not _lib.stream_done(side, event) and _lib.stream_done(torch.cuda.default_stream())
    again.replay()
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want) and torch.equal(layer(x), want)
