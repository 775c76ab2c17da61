"""A layer that is called on several streams and from several threads: the forms of its weight that the first call builds on its own stream are whole
for every other."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _make(family, layer_type, w, backend="fused"):
    import mase_hip.minifloat.meta as mf
    import mase_hip.mxfp.meta as mx
    from mase_hip.minifloat.layers import MinifloatLinearPTQ
    from mase_hip.mxfp.layers import MXFPLinearPTQ

    if family == "mxfp":
        return MXFPLinearPTQ(w, None, mx.MXFP8_E4M3_fn if layer_type == "XqWqB" else None, mx.OCP_MXFP4_E2M1, None, layer_type, backend)
    return MinifloatLinearPTQ(weight=w, bias=None, x_minifloat_meta=mf.FP8_E4M3_fn if layer_type == "XqWqB" else None, w_minifloat_meta=mf.FP4_E2M1_fn,
                              b_minifloat_meta=None, layer_type=layer_type, backend=backend)


CASES = [("XqWqB", 48), ("XqWqB", 2000), ("XWqB", 12), ("XWqB", 3000)]     # the packed and the block-scaled form, packed for dense rows, prepared


@pytest.mark.parametrize("family", ["mxfp", "minifloat"])
@pytest.mark.parametrize("layer_type,rows", CASES)
def test_forms_built_behind_other_work_of_their_stream(family, layer_type, rows):
    K, N = 4096, 2048
    g = torch.Generator(device=DEV).manual_seed(rows)
    w, w2 = ((0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16) for _ in range(2))
    x = torch.randn(rows, K, generator=g, device=DEV).to(torch.bfloat16)
    busy = torch.randn(4096, 4096, generator=g, device=DEV)
    layer, warm, other = _make(family, layer_type, w), _make(family, layer_type, w), _make(family, layer_type, w2)
    want, want2 = warm(x), other(x)
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    for i, expect in ((0, want), (1, want2)):
        if i:
            layer.load_state_dict(other.state_dict())                       # new forms in the place of old ones
            torch.cuda.synchronize()
        outs = []
        for s in streams:
            with torch.cuda.stream(s):
                if s is streams[0]:
                    for _ in range(20):
                        torch.mm(busy, busy)
                outs.append(layer(x))
        torch.cuda.synchronize()
        assert all(torch.equal(y, expect) for y in outs)


@pytest.mark.parametrize("family", ["mxfp", "minifloat"])
def test_forms_built_on_a_stream_of_another_owner(family):
    """No later call asks anything of such a stream, which may be gone by then."""
    g = torch.Generator(device=DEV).manual_seed(3)
    w = (0.5 * torch.randn(2048, 4096, generator=g, device=DEV)).to(torch.bfloat16)
    x = torch.randn(48, 4096, generator=g, device=DEV).to(torch.bfloat16)
    layer, warm = _make(family, "XqWqB", w), _make(family, "XqWqB", w)
    want, own = warm(x), torch.cuda.Stream()
    torch.cuda.synchronize()
    assert warm._packed_w.stream is not None
    with torch.cuda.stream(torch.cuda.ExternalStream(own.cuda_stream)):
        y = layer(x)
    assert layer._packed_w.stream is None and (layer._scaled_w is None) == (warm._scaled_w is None)
    with torch.cuda.stream(own):
        z = layer(x)
    torch.cuda.synchronize()
    assert torch.equal(y, want) and torch.equal(z, want)


@pytest.mark.parametrize("family", ["mxfp", "minifloat"])
def test_threads_with_streams_of_their_own(family):
    """Decode-sized and prefill-sized calls of the same fresh layers, each thread with its own mix."""
    K, N, rows = 4096, 2048, (1, 12, 48, 600, 3000)
    g = torch.Generator(device=DEV).manual_seed(5)
    xs = [torch.randn(r, K, generator=g, device=DEV).to(torch.bfloat16) for r in rows]
    for layer_type in ("XqWqB", "XWqB"):
        w = (0.5 * torch.randn(N, K, generator=g, device=DEV)).to(torch.bfloat16)
        warm = _make(family, layer_type, w)
        want = [warm(x) for x in xs]
        for _ in range(5):
            layer, bad = _make(family, layer_type, w), []
            torch.cuda.synchronize()

            def calls(first):
                try:
                    with torch.cuda.stream(torch.cuda.Stream()):
                        ys = [(i, layer(xs[i])) for k in range(10) for i in [(first + k * (first + 1)) % len(xs)]]
                        torch.cuda.current_stream().synchronize()
                    bad.extend(rows[i] for i, y in ys if not torch.equal(y, want[i]))
                except Exception as e:      # noqa: BLE001
                    bad.append(repr(e))

            threads = [threading.Thread(target=calls, args=(t,)) for t in range(4)]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            assert not bad, (layer_type, bad)
