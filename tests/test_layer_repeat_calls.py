"""What a layer remembers of its last call: nothing of a call that failed, nothing across a move, and no more than an older pickle holds."""
import pytest
import torch

import mase_hip.minifloat.functional as MF
import mase_hip.mxfp.functional as MX
from mase_hip.minifloat.layers import MinifloatLinearPTQ
from mase_hip.mxfp.layers import MXFPLinearPTQ


@pytest.fixture(params=["mxfp", "minifloat"])
def layer_and_calls(request, monkeypatch):
    """A weightless layer whose product and weight operand are stand-ins: calls of the operand rule, and a switch that makes the product fail."""
    calls = {"asked": 0, "fail": False}

    def ask(self, input):
        calls["asked"] += 1

    def product(**kw):
        if calls["fail"]:
            raise RuntimeError("refused")
        return kw["x"]

    if request.param == "mxfp":
        cls, mod, name = MXFPLinearPTQ, MX, "mxfp_linear"
        layer = cls(weight=torch.zeros(32, 32), bias=None, x_mxfp_meta=None, w_mxfp_meta=None, b_mxfp_meta=None, layer_type="XW", backend="separate")
    else:
        cls, mod, name = MinifloatLinearPTQ, MF, "minifloat_linear"
        layer = cls(weight=torch.zeros(32, 32), bias=None, x_minifloat_meta=None, w_minifloat_meta=None, b_minifloat_meta=None, layer_type="XW",
                    backend="separate")
    monkeypatch.setattr(cls, "_weight_operand", ask)
    monkeypatch.setattr(mod, name, product)
    return layer, calls


def test_repeat_is_not_asked_about(layer_and_calls):
    layer, calls = layer_and_calls
    for rows, asked in ((2, 1), (2, 1), (3, 2), (2, 3)):
        layer(torch.zeros(rows, 32))
        assert calls["asked"] == asked


def test_failed_call_is_forgotten(layer_and_calls):
    layer, calls = layer_and_calls
    calls["fail"] = True
    for asked in (1, 2):
        with pytest.raises(RuntimeError, match="refused"):
            layer(torch.zeros(2, 32))
        assert calls["asked"] == asked


def test_move_and_older_pickle(layer_and_calls):
    layer, calls = layer_and_calls
    layer(torch.zeros(2, 32))
    layer.to("cpu")
    layer(torch.zeros(2, 32))
    assert calls["asked"] == 2
    layer.__dict__.pop("_no_operand_sig")
    layer(torch.zeros(2, 32))
    assert calls["asked"] == 3


def test_notes_cost_no_module_assignments(layer_and_calls, monkeypatch):
    """A call notes what it was without nn.Module's own assignment (1 - 2 us each: calls of changing row counts took 9.0 us of host time
    before there were notes and 13.4 with two more assignments, 8.2 now)."""
    layer, calls = layer_and_calls
    names = []
    assign = type(layer).__setattr__
    monkeypatch.setattr(type(layer), "__setattr__", lambda self, name, value: (names.append(name), assign(self, name, value))[1])
    for rows in (2, 3, 3, 2):
        layer(torch.zeros(rows, 32))
    assert names == [] and calls["asked"] == 3
    assert layer._no_operand_sig is not None and layer._fast_sig is None


def test_what_a_call_is_not_eligible_for_is_not_asked_again(layer_and_calls, monkeypatch):
    """Calls that the extension does not take (fp16, a format that the kernels do not decode) are looked at once for every look."""
    import mase_hip.minifloat.functional.linear as MFL
    import mase_hip.mxfp.functional.linear as MXL

    layer, calls = layer_and_calls
    asked = []
    for L in (MXL, MFL):
        monkeypatch.setattr(L, "_gemm_eligible", lambda *a: asked.append(1))
    layer.layer_type, layer.backend = "XqWq", "fused"
    layer.w_tensor_meta = None
    for rows, times in ((2, 1), (2, 1), (2, 1), (3, 2), (2, 3), (2, 3)):
        layer(torch.zeros(rows, 32))
        assert len(asked) == times and layer._fast_sig is None
