"""The other forms of a quantised weight that a layer keeps, with stand-ins for the kernels that build and read them: what becomes of them when the
components move or change."""
import pytest
import torch

import mase_hip.mxfp.functional as MX
import mase_hip.mxfp.meta as mx
from mase_hip.mxfp import kernels
from mase_hip.mxfp.layers import MXFPLinearPTQ

N, K = 2048, 4096        # (freshly mapped pages, which an allocator hands out again at once)


def components(seed, dtype=torch.uint8):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, 16, (N * K // 32, 1), generator=g, dtype=dtype), torch.randint(0, 16, (N * K // 32, 32), generator=g, dtype=dtype)


class Form:
    """What a stand-in builds: the sum of the codes that it was given."""

    def __init__(self, elements):
        self.sum = int(elements.sum(dtype=torch.int64))


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr("mase_hip.mxfp.functional.linear.scaled_weight_operand", lambda scales, elements, meta: Form(elements))
    monkeypatch.setattr(kernels, "packed_weight_from_mxfp", lambda scales, elements, e, m, rows, k: Form(elements))
    monkeypatch.setattr(kernels, "packed_pays", lambda *a: True)
    scales, elements = components(0)
    meta = mx.MXFPTensorMeta(device="cpu", dtype="bfloat16", shape=(N, K), block_dim=1, meta=mx.OCP_MXFP4_E2M1)
    return MXFPLinearPTQ.from_quantized(scales, elements, meta, None, None, None, None, mx.MXFP8_E4M3_fn, "XqWqB", "fused")


class OnGpu:
    """As much of an input on a GPU as the rules ask for."""

    device, dtype, shape = torch.device("cuda", 0), torch.bfloat16, torch.Size((4, K))

    def numel(self):
        return 4 * K


def both_forms(layer):
    return layer._prepared_weight(), layer._packed_weight(OnGpu(), True)[0]


def test_forms_go_with_the_components_that_move(layer):
    both_forms(layer)
    assert layer._scaled_w is not None and layer._packed_w is not None
    kept = layer._scaled_w, layer._packed_w
    layer.to("cpu")                                    # nothing moves
    assert (layer._scaled_w, layer._packed_w) == kept
    layer.to("meta")
    assert layer._scaled_w is None and layer._packed_w is None
