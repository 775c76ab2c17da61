"""The further forms of a quantised weight that a layer keeps, with stand-ins for the kernels that build and read them: what becomes of them when the
components move or change."""
import copy
import dataclasses
import pickle

import pytest
import torch
import torch.nn.utils.parametrize

import mase_hip.mxfp.functional as MX
import mase_hip.mxfp.meta as mx
from mase_hip import _lib
from mase_hip.mxfp import kernels
from mase_hip.mxfp.layers import MXFPLinearPTQ
from mase_hip.utils import qlayer

N, K = 2048, 4096        # (freshly mapped pages, which an allocator hands out again at once)


def components(seed, dtype=torch.uint8):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(0, 16, (N * K // 32, 1), generator=g, dtype=dtype), torch.randint(0, 16, (N * K // 32, 32), generator=g, dtype=dtype)


class Form:
    """What a stand-in builds: the sum of the codes that it was given."""

    codes = scales = exp_bits = frac_bits = None

    def __init__(self, elements, into=None):
        self.memory = object() if into is None else into.memory
        self.sum = int(elements.sum(dtype=torch.int64))


@pytest.fixture
def layer(monkeypatch):
    monkeypatch.setattr("mase_hip.mxfp.functional.linear.scaled_weight_operand", lambda scales, elements, meta, into: Form(elements, into))
    monkeypatch.setattr(kernels, "packed_weight_from_mxfp", lambda scales, elements, e, m, rows, k, into: Form(elements, into))
    monkeypatch.setattr(kernels, "packed_pays", lambda *a: True)
    scales, elements = components(0)
    meta = mx.MXFPTensorMeta(device="cpu", dtype="bfloat16", shape=(N, K), block_dim=1, meta=mx.OCP_MXFP4_E2M1)
    return MXFPLinearPTQ.from_quantized(scales, elements, meta, None, None, None, None, mx.MXFP8_E4M3_fn, "XqWqB", "fused")


class OnGpu:
    """As much of an input on a GPU as the rules ask for."""

    device, dtype, shape = torch.device("cuda", 0), torch.bfloat16, torch.Size((4, K))

    def numel(self):
        return 4 * K

    def reshape(self, *shape):
        return self


def both_forms(layer):
    return layer._weight_form("_scaled_w"), layer._weight_form("_packed_w")


def test_forms_go_with_the_components_that_move(layer):
    both_forms(layer)
    assert layer._scaled_w is not None and layer._packed_w is not None
    kept = layer._scaled_w, layer._packed_w
    layer.to("cpu")                                    # nothing moves
    assert (layer._scaled_w, layer._packed_w) == kept
    layer.to("meta")
    assert layer._scaled_w is None and layer._packed_w is None


def test_components_at_a_former_address_are_not_the_former_components(layer):
    """A freed component's memory goes to the next one of its size, whose version is 0 again."""
    seen = set()
    for seed in range(1, 30):
        assert [f.value.sum for f in both_forms(layer)] == [int(layer.w_elements.sum(dtype=torch.int64))] * 2
        seen.add(layer._scaled_w.key)
        layer.w_elements = layer.w_scales = None
        scales, elements = components(seed)
        layer.w_scales, layer.w_elements = (torch.nn.Parameter(t, requires_grad=False) for t in (scales, elements))
    assert len(seen) > 1


def test_a_copy_builds_its_own_forms(layer):
    both_forms(layer)
    for other in (copy.deepcopy(layer), pickle.loads(pickle.dumps(layer))):
        assert other._scaled_w is None and other._packed_w is None and layer._scaled_w is not None
    state = layer.__getstate__()
    state.update(_scaled_w=object(), _fast_sig=(), _fast_packed=1)      # as a layer was pickled that kept forms without their components
    other = MXFPLinearPTQ.__new__(MXFPLinearPTQ)
    other.__setstate__(state)
    assert other._scaled_w is None and other._fast_sig is None


def test_forms_built_for_a_graph_are_not_kept(layer, monkeypatch):
    """What a captured stream is given runs on the replays: nothing is written yet for the calls between."""
    monkeypatch.setattr(qlayer, "capturing", lambda device: True)
    assert layer._packed_weight(OnGpu(), True) is qlayer.NOT_NOW and layer._weight_form("_scaled_w").value.sum > 0
    assert layer._scaled_w is None and layer._packed_w is None
    monkeypatch.setattr(qlayer, "capturing", lambda device: False)
    kept = both_forms(layer)
    monkeypatch.setattr(qlayer, "capturing", lambda device: True)
    assert both_forms(layer) == kept == (layer._scaled_w, layer._packed_w)


def test_only_calls_that_have_a_use_for_a_form_ask_about_captures(layer, monkeypatch):
    """fp16 calls, and those of many rows on the components, whatever their shape was last; of the others a captured one that went without is not noted."""
    layer.layer_type, layer.x_mxfp_meta, asked = "XWqB", None, []
    monkeypatch.setattr(qlayer, "capturing", lambda device: asked.append(device) or True)
    monkeypatch.setattr(kernels, "packed_dense_pays", lambda rows, *a: rows <= 32)
    monkeypatch.setattr(kernels, "prepared_w_pays", lambda rows, *a: rows >= 1000)
    monkeypatch.setattr(OnGpu, "numel", lambda self: self.shape.numel())
    monkeypatch.setattr(MX, "mxfp_linear", lambda **kw: torch.zeros(1))
    for rows, dtype, has_use in ((4, torch.float16, False), (8, torch.float16, False), (40, torch.bfloat16, False), (60, torch.bfloat16, False), (4, torch.bfloat16, True),
                                 (1000, torch.bfloat16, True)):
        x = OnGpu()
        x.shape, x.dtype = torch.Size((rows, K)), dtype
        asked.clear()
        layer(x)
        assert bool(asked) == has_use and (layer._no_operand_sig is None) == has_use


def test_a_layer_that_is_given_a_weight_of_another_format(layer, monkeypatch):
    """Neither the way of the last call nor a form outlives what the codes meant then."""
    kept, taken = both_forms(layer), []
    layer.w_tensor_meta = layer.w_tensor_meta.create(meta=mx.OCP_MXFP6_E3M2)
    assert not set(both_forms(layer)) & set(kept) and layer._scaled_w.format is mx.OCP_MXFP6_E3M2
    kept = both_forms(layer)
    layer.w_tensor_meta = layer.w_tensor_meta.create(meta=dataclasses.replace(mx.OCP_MXFP6_E3M2))       # the same, another object
    assert both_forms(layer) == kept

    class Host:
        linear_plain = staticmethod(lambda *a: taken.append(a[5:7]) or torch.zeros(4, N))

    monkeypatch.setattr(_lib, "_host", Host)
    monkeypatch.setattr(kernels, "packed_dense_pays", lambda *a: False)
    monkeypatch.setattr(kernels, "prepared_w_pays", lambda *a: False)
    monkeypatch.setattr("mase_hip.mxfp.functional.linear._gemm_eligible", lambda x, quantised, tm, b: tm.meta.element_is_finite)
    monkeypatch.setattr(MX, "mxfp_linear", lambda **kw: torch.zeros(4, N))
    layer.layer_type, layer.x_mxfp_meta = "XWqB", None
    for _ in range(3):
        layer(OnGpu())
    assert taken == [(3, 2)] * 2
    scales, elements = components(1)
    layer.w_scales, layer.w_elements = (torch.nn.Parameter(t, requires_grad=False) for t in (scales, elements))
    layer.w_tensor_meta = layer.w_tensor_meta.create(meta=mx.MXFPMeta(32, 8, 5, 2, False, "rn"))        # its top exponent field is inf / NaN, which the kernels do not know
    for _ in range(3):
        layer(OnGpu())
    assert len(taken) == 2


class Stream:
    """A stand-in for a stream on a GPU: the events recorded on it, and those that it waits for."""

    def __init__(self, number):
        self.cuda_stream, self.recorded, self.waits, self.done, self.captured = number, [], [], False, False

    def __getitem__(self, i):      # (as torch names it: its number, its device, ..)
        return self.cuda_stream * 2 + 1

    def record_event(self):
        self.recorded.append(Event())
        return self.recorded[-1]

    def wait_event(self, event):
        self.waits.append(event)


class Event:
    done = False


def test_calls_go_behind_what_writes_a_form(layer, monkeypatch):
    """Calls on the stream that the form is written on have the order; of others each waits for an event of that stream, until one is found to have run."""
    a, b, products = Stream(1), Stream(2), []
    at = [a]
    monkeypatch.setattr(_lib, "dense", lambda t: t)
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: at[0].cuda_stream)
    monkeypatch.setattr(_lib, "stream_done", lambda stream, event=None: (stream if event is None else event).done and not stream.captured)
    monkeypatch.setattr(qlayer, "current_stream", lambda device: at[0])
    monkeypatch.setattr(qlayer, "as_stream", lambda name: name)
    monkeypatch.setattr(qlayer, "capturing", lambda device: at[0].captured)
    monkeypatch.setattr(qlayer, "stream_captured", lambda stream: stream.captured)
    monkeypatch.setattr(qlayer.torch.cuda, "current_stream", lambda device: at[0])
    monkeypatch.setattr(kernels, "linear_packed", lambda *args: (products.append("wrappers"), torch.zeros(4, N))[1])

    class Host:
        linear_packed = staticmethod(lambda *args: products.append("extension") or (torch.zeros(4, N) if takes else None))

    def build(written=False):
        layer._drop_forms()
        layer(OnGpu())
        if written:
            a.done = True
        return layer._packed_w

    takes = False
    monkeypatch.setattr(_lib, "_host", Host)
    form = build()
    assert form.stream is a and not a.recorded and products == ["extension", "wrappers"]
    takes = True
    # another stream first: the event is recorded there and then, on the form's stream
    at[0] = b
    layer(OnGpu())
    layer._forward(OnGpu(), ())
    assert len(a.recorded) == 1 and b.waits == a.recorded * 2 and not b.recorded and products[2:] == ["extension"] * 2
    at[0] = a
    layer(OnGpu())
    assert not a.waits and form.stream is a
    a.recorded[0].done = True
    at[0] = b
    layer(OnGpu())
    assert form.stream is None and len(b.waits) == 2 and len(a.recorded) == 1
    # its own stream first
    at[0] = a
    form = build()
    layer(OnGpu())
    assert form.event is a.recorded[1] and not a.waits
    # captured calls: one on another stream asks the form's stream or its event, one on the form's own only the event
    b.captured, at[0] = True, b
    assert layer._packed_weight(OnGpu(), True) is qlayer.NOT_NOW and len(b.waits) == 2
    a.recorded[1].done = True
    assert layer._packed_weight(OnGpu(), True)[0] is form.value and layer._packed_w is form and form.stream is None
    at[0] = a
    form = build()
    at[0] = b
    assert layer._packed_weight(OnGpu(), True) is qlayer.NOT_NOW and layer._packed_w is form
    a.done = True
    assert layer._packed_weight(OnGpu(), True)[0] is form.value and layer._packed_w is form and form.stream is None and len(a.recorded) == 2
    at[0], a.done = a, False
    form = build(written=True)
    a.captured = True
    assert layer._packed_weight(OnGpu(), True) is qlayer.NOT_NOW
    # an eager call while the form's stream is captured by another thread: a form of its own
    b.captured, at[0] = False, b
    other = layer._packed_weight(OnGpu(), True)[0]
    assert layer._packed_w is form and other.memory is not form.value.memory and len(a.recorded) == 2
    # written in place: in the same memory, behind what wrote it before
    a.captured = False
    with torch.no_grad():
        layer.w_elements.add_(1)
    layer._forward(OnGpu(), ())
    assert b.waits[-1] is a.recorded[2] and layer._packed_w is not form and layer._packed_w.value.memory is form.value.memory and layer._packed_w.stream is b


def test_no_event_is_recorded_on_a_stream_that_its_owner_may_have_destroyed(layer, monkeypatch):
    """The call that builds a form on a stream that torch was handed waits for it."""
    waited = []

    class External:
        synchronize = staticmethod(lambda: waited.append("stream"))

        def __getattr__(self, name):
            raise AssertionError(name)

    at = [(0x55550010, 0, 1)]
    monkeypatch.setattr(qlayer, "current_stream", lambda device: at[0])
    monkeypatch.setattr(qlayer, "as_stream", lambda name: External())
    form = layer._weight_form("_packed_w")
    assert waited == ["stream"] and form.stream is None and layer._weight_form("_packed_w") is form
    for at[0] in ((0, 0, 1), (0x23, 0, 1), None):                 # torch's own
        layer._drop_forms()
        assert layer._weight_form("_packed_w").stream == at[0] and len(waited) == 1


def test_of_two_threads_that_build_a_form_one_keeps_its_own(layer, monkeypatch):
    """The other uses what it has built: a form that calls on other streams may already read is not given back."""
    build, first = layer._build_form, []

    def build_and_be_overtaken(name, into, *components):
        if not first:
            first.append(None)
            first.append(layer._weight_form(name))
        return build(name, into, *components)

    monkeypatch.setattr(layer, "_build_form", build_and_be_overtaken)
    form = layer._weight_form("_scaled_w")
    assert layer._scaled_w is first[1] is not form and form.value.sum == first[1].value.sum


def test_components_that_a_parametrisation_makes_have_no_kept_forms(layer):
    class Same(torch.nn.Module):
        def forward(self, t):
            return t.clone()

    torch.nn.utils.parametrize.register_parametrization(layer, "w_elements", Same(), unsafe=True)
    for delta in (0, 1, 1):
        layer.parametrizations.w_elements.original.data.add_(delta)
        assert [f.value.sum for f in both_forms(layer)] == [int(layer.w_elements.sum(dtype=torch.int64))] * 2
        assert layer._scaled_w is None and layer._packed_w is None


def test_a_call_between_the_steps_of_another(layer, monkeypatch):
    """A weight-only layer shared by a prefill and a decode thread: a decode call that lands where the prefill call asks for its route."""
    layer.layer_type, layer.x_mxfp_meta = "XWqB", None
    small, large, taken = OnGpu(), OnGpu(), []
    large.shape = torch.Size((600, K))

    class Host:
        linear_packed_dense = staticmethod(lambda *a: taken.append("dense") or torch.zeros(4, N))

    monkeypatch.setattr(_lib, "_host", Host)
    monkeypatch.setattr(kernels, "packed_dense_pays", lambda rows, *a: rows <= 32)
    monkeypatch.setattr(kernels, "mxfp_gemm_packed_dense", lambda *a: torch.zeros(4, N))
    monkeypatch.setattr(kernels, "prepared_w_shape_supported", lambda *a: True)
    monkeypatch.setattr(kernels, "prepared_w_pays", lambda *a: True)
    monkeypatch.setattr(MX, "mxfp_linear", lambda **kw: torch.zeros(600, N))
    monkeypatch.setattr(OnGpu, "numel", lambda self: self.shape.numel())
    layer(large)                                      # both forms are there
    layer(small)
    asked = MXFPLinearPTQ._takes_scaled_route
    monkeypatch.setattr(MXFPLinearPTQ, "_takes_scaled_route", lambda self, x: asked(self, x) if x is small else (layer(small), asked(self, x))[1])
    layer(large)
    assert taken and set(taken) == {"dense"}


def test_what_a_graph_reads_follows_components_written_in_place(layer, monkeypatch):
    """A captured call reads the kept forms where they lie: a form of new values takes the memory of the one that it replaces, unless the components are others."""
    before = [f.value.memory for f in both_forms(layer)]
    state = {k: v + 1 for k, v in layer.state_dict().items()}
    layer.load_state_dict(state)                                 # (without a call behind it)
    forms = layer._scaled_w.value, layer._packed_w.value
    assert [f.memory for f in forms] == before and [f.sum for f in forms] == [int(state["w_elements"].sum(dtype=torch.int64))] * 2
    with torch.no_grad():
        layer.w_elements.sub_(1)
    assert [f.value.memory for f in both_forms(layer)] == before
    monkeypatch.setattr(qlayer, "capturing", lambda device: True)
    with torch.no_grad():
        layer.w_elements.add_(1)
    assert layer._weight_form("_scaled_w").value.memory not in before                # (a graph's own form)
    monkeypatch.setattr(qlayer, "capturing", lambda device: False)
    layer.load_state_dict(state, assign=True)
    assert not set(f.value.memory for f in both_forms(layer)) & set(before)


def test_no_form_is_built_that_the_call_does_not_read(layer, monkeypatch):
    """A weight-only call of many rows whose product is faster on the components."""
    layer.layer_type, layer.x_mxfp_meta = "XWqB", None
    monkeypatch.setattr(kernels, "prepared_w_shape_supported", lambda *a: True)
    for pays in (False, True):
        monkeypatch.setattr(kernels, "prepared_w_pays", lambda *a: pays)
        assert (layer._weight_operand(OnGpu()) is not None) == pays


def test_layers_of_inference_tensors_move_and_load(layer):
    """Their components have no versions."""
    with torch.inference_mode():
        scales, elements = components(1)
        made = MXFPLinearPTQ.from_quantized(scales, elements, layer.w_tensor_meta, None, None, None, None, None, "XWqB", "fused")
        assert made.w_elements.is_inference() and made.to("cpu") is made
        made.load_state_dict(layer.state_dict())
        assert torch.equal(made.w_elements, layer.w_elements)
        both_forms(layer)
        layer.w_scales, layer.w_elements = made.w_scales, made.w_elements       # forms of what it had before
        layer.load_state_dict(layer.state_dict())
        layer.to("cpu")
        assert layer._scaled_w is None and layer._packed_w is None


def test_weight_only_calls_read_components_whose_writes_are_not_counted(layer, monkeypatch):
    """A layer that was moved in inference mode, and one that was built in it: a packed form would not follow a write in place."""
    monkeypatch.setattr(kernels, "packed_dense_pays", lambda *a: True)
    layer.layer_type, layer.x_mxfp_meta = "XWqB", None
    assert layer._packed_weight(OnGpu())[1]
    with torch.inference_mode():
        for name in ("w_scales", "w_elements"):
            getattr(layer, name).data = getattr(layer, name).clone()
        before = layer.w_elements._version
        layer.w_elements.add_(1)
        assert layer.w_elements._version == before and layer._packed_weight(OnGpu()) is None
        scales, elements = components(1)
        made = MXFPLinearPTQ.from_quantized(scales, elements, layer.w_tensor_meta, None, None, None, None, None, "XWqB", "fused")
        assert made._packed_weight(OnGpu()) is None


@pytest.mark.parametrize("built_in,written_in", [(True, False), (False, True), (True, True), (False, False)])
def test_narrowed_codes_are_written_again_in_either_mode(built_in, written_in):
    """Codes that a call in inference mode built, written again by one outside of it, and the other way round."""
    import mase_hip.minifloat.functional as MF
    import mase_hip.minifloat.meta as mf

    meta = mf.MinifloatTensorMeta(device="cpu", dtype="bfloat16", shape=(4, 64), meta=mf.FP6_E3M2_fn)
    first, second = (torch.randint(0, 64, (4, 64), dtype=torch.int16).view(torch.uint16) for _ in range(2))
    with torch.inference_mode(built_in):
        kept = MF.narrow_weight_codes(first, meta)
    at = kept[1].data_ptr()
    with torch.inference_mode(written_in), torch.no_grad():
        again = MF.narrow_weight_codes(second, meta, kept)
    assert again[1].data_ptr() == at and torch.equal(again[1].to(torch.int16), second.view(torch.int16))
