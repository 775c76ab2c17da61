"""Helpers for the PTQ layers (the first two: same contract as src/mase_triton/utils/qlayer.py:4-21)."""
import threading

import torch

from .. import _lib


class ChangeDtypeError(Exception):
    """Raised when ``.to(dtype=...)`` would change the dtype of stored integer codes."""

    def __init__(self, message="Changing dtype is not allowed."):
        self.message = message
        super().__init__(message)


def _canonical(device) -> torch.device:
    d = torch.device(device)
    return torch.device("cuda", 0) if d.type == "cuda" and d.index is None else d


def devices_equal(device1, device2) -> bool:
    """True if both name the same device; a bare "cuda" means "cuda:0"."""
    return _canonical(device1) == _canonical(device2)


def weight_key(components) -> tuple:
    """Address and version of each.  (Tensors made in inference mode have no version; asking for it raises.)"""
    key = ()
    for c in components:
        key += (c.data_ptr(), c._version)
    return key


def capturing(device: torch.device) -> bool:
    """Is the current stream of ``device`` being captured into a graph?  (What is launched then runs when the graph does, not now.)"""
    if device.type != "cuda":
        return False
    with _lib.on_device(device):
        return torch.cuda.is_current_stream_capturing()


def stream_captured(stream) -> bool:
    with torch.cuda.stream(stream):
        return torch.cuda.is_current_stream_capturing()


def current_stream(device: torch.device):
    """What names the stream that a form built now is written on (None: nothing runs behind the host)."""
    return torch._C._cuda_getCurrentStream(device.index) if device.type == "cuda" else None


def as_stream(name) -> "torch.cuda.Stream":
    stream_id, device_index, device_type = name
    return torch.cuda.Stream(stream_id=stream_id, device_index=device_index, device_type=device_type)


def owned_elsewhere(name) -> bool:
    """Is it a stream that torch was handed (``ExternalStream``), whose owner may destroy it?  (torch's own are never destroyed; their numbers are odd, and
    0 for the default one, where a stream of another owner is named by its handle.)"""
    return name is not None and name[0] != 0 and name[0] % 2 == 0


# What a layer answers where a call has a use for a form that the graph which is being captured cannot read yet.  (Asking the stream instead whether it is
# captured took 2 us of the 20 that a call of another row count than the last one's takes the host.)
NOT_NOW = ()


class WeightForm:
    """A quantised weight in another form than its stored components.

    ``key`` names the components that it was built from, by address and version.  An address names a tensor only until its memory is handed out
    again, so the form holds the memory of each: whatever replaces a component while the form is kept lies elsewhere.  ``format`` is what their codes meant.  ``stream`` names the one that the
    kernels which write the form were launched on, None once they are known to have run; ``event`` is behind them, once one was asked for."""

    __slots__ = ("value", "key", "format", "memory", "device", "stream", "event")

    def __init__(self, value, key: tuple, format, components, stream):
        self.value, self.key, self.format, self.memory, self.device = value, key, format, [c.untyped_storage() for c in components], components[0].device
        self.stream, self.event = stream, None

    def ready(self) -> bool:
        """Put the current stream behind what writes the form; False where that cannot be: one of the two is captured and the form not known to be written.

        The building call records no event (it costs the host 6 us, and the next kernel waits behind it: the first call of a SwiGLU block of two layers, 6 x
        1024 x 4096, took 139 us without and 159 with); the first call behind it does, on the form's stream, whichever its own is."""
        stream, device = self.stream, self.device
        if stream is None:
            return True
        stream = as_stream(stream)
        event, own, captured = self.event, _lib.stream_ptr(device) == stream.cuda_stream, capturing(device)
        if (event is not None or captured) and _lib.stream_done(stream, event):
            self.stream = None
            return True
        if event is None and not captured:
            if not own and stream_captured(stream):
                return False
            event = self.event = stream.record_event()
        if captured:
            return False
        if not own:
            with _lib.on_device(device):
                torch.cuda.current_stream(device).wait_event(event)
        return True


_publish = threading.Lock()


class KeepsWeightForms:
    """What the PTQ layers have in common that keep their weight in further forms (attributes named by ``_FORMS``) beside the components
    (``_FORM_COMPONENTS``).  Forms are built on the first call that reads them and again after a change of the components, and are part of
    neither ``state_dict`` nor a copy or pickle of the layer.

    A form is built on the stream of one call and read by calls on any stream and of any thread, which go behind what writes it until that is known to
    have run (``WeightForm.ready``).  (The building call could wait for its stream instead: a new layer's first call 63 -> 93 us.)

    A captured call reads the forms that were kept then, where they lie.  So components that are written in place are built into the same memory again,
    by the next call or by ``load_state_dict`` itself, and replays follow; a graph is captured again after the components were replaced or moved or
    ``invalidate_weight_operand`` was called."""

    _FORMS: tuple[str, ...] = ()
    _FORM_COMPONENTS: tuple[str, ...] = ()
    # What the last call looked like that a call of the same look may follow without the checks, and the way that it went.  One tuple, read once and
    # written once: a thread's call can lie between any two steps of another's.
    _note: tuple[tuple, int] | None = None

    @property
    def _fast_sig(self):
        return None if (note := self._note) is None else note[0]

    @property
    def _fast_packed(self) -> int:
        return 0 if (note := self._note) is None else note[1]

    def _build_form(self, name: str, into, *components: torch.Tensor):
        """The value of form ``name``, in the memory of the value ``into`` if that is given."""
        raise NotImplementedError

    def _weight_form(self, name: str, needed: bool = True) -> WeightForm | None:
        """The form ``name`` of the weight as it is now, for the current stream.  One that is built while the stream is captured belongs to that graph, which
        writes it on every replay; with ``needed`` false, for a call that has another way, None in its place."""
        held = self._parameters
        components = [held[c] if held.get(c) is not None else getattr(self, c) for c in self._FORM_COMPONENTS]
        kept, key, device, format = getattr(self, name), weight_key(components), components[0].device, self.w_tensor_meta.meta
        same = kept is not None and kept.key == key and (kept.format is format or kept.format == format)
        if same and kept.ready():
            return kept
        in_graph = capturing(device)
        if in_graph and not needed:
            return None
        # (the same, which this stream cannot be put behind; or the same tensors, written since or of another format)
        written = not same and kept is not None and kept.key[::2] == key[::2] and not in_graph and kept.ready()
        stream = None if in_graph else current_stream(device)
        form = WeightForm(self._build_form(name, kept.value if written else None, *components), key, format, components, stream)
        if owned_elsewhere(stream):                           # (it may be gone when the next call would record an event on it)
            as_stream(stream).synchronize()
            form.stream = None
        if in_graph or same or self._computed_components():
            return form
        if kept is not None and not written and device.type == "cuda":
            torch.cuda.synchronize(device)                    # (calls on other streams may still read the one that goes)
        with _publish:
            if getattr(self, name) is kept:                   # (else another thread's call was faster)
                self.__dict__[name] = form
        return form

    def _computed_components(self) -> bool:
        """Does a parametrisation make the components anew for every call?"""
        cls = type(self)
        for c in self._FORM_COMPONENTS:
            if isinstance(getattr(cls, c, None), property):
                return True
        return False

    def _drop_forms(self, moved_only: bool = False) -> None:
        """Forget the forms, or those whose components are not the layer's any more."""
        addresses = self._component_addresses()
        for name in self._FORMS:
            kept = getattr(self, name)
            if kept is not None and not (moved_only and kept.key[::2] == addresses):
                self.__dict__[name] = self.__dict__["_note"] = None

    def _component_addresses(self) -> tuple:
        components = [getattr(self, c) for c in self._FORM_COMPONENTS]
        return tuple(None if c is None else c.data_ptr() for c in components)

    def _load_from_state_dict(self, *args, **kwargs):
        super()._load_from_state_dict(*args, **kwargs)
        for name in self._FORMS:
            kept = getattr(self, name)
            if kept is not None and kept.key[::2] == self._component_addresses():
                self._weight_form(name)

    def __getstate__(self):
        return {**self.__dict__, **dict.fromkeys(self._FORMS), "_note": None}

    def __setstate__(self, state):
        super().__setstate__({**state, **dict.fromkeys(self._FORMS), "_note": None})         # (older pickles hold forms without a key)
