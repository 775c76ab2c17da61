"""Helpers for the PTQ layers (the first two: same contract as src/mase_triton/utils/qlayer.py:4-21)."""
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


class WeightForm:
    """A quantised weight in another form than its stored components.

    ``key`` names the components that it was built from, by address and version.  An address names a tensor only until its memory is handed out
    again, so the form holds an alias of each: whatever replaces a component while the form is kept lies elsewhere."""

    __slots__ = ("value", "key", "components")

    def __init__(self, value, key: tuple, components: tuple):
        self.value, self.key, self.components = value, key, components


def weight_key(components) -> tuple:
    return tuple(v for c in components for v in (c.data_ptr(), c._version))


def capturing(device: torch.device) -> bool:
    """Is the current stream of ``device`` being captured into a graph?  (What is launched then runs when the graph does, not now.)"""
    if device.type != "cuda":
        return False
    with _lib.on_device(device):
        return torch.cuda.is_current_stream_capturing()


def finish(device: torch.device, every_stream: bool) -> None:
    """Wait for the current stream of ``device``, or for all its streams."""
    with _lib.on_device(device):
        torch.cuda.synchronize(device) if every_stream else torch.cuda.current_stream(device).synchronize()


class KeepsWeightForms:
    """What the PTQ layers have in common that keep their weight in further forms (attributes named by ``_FORMS``) beside the components
    (``_FORM_COMPONENTS``).  Forms are built on the first call that reads them and again after a change of the components, and are part of
    neither ``state_dict`` nor a copy or pickle of the layer.

    A form is built on the stream of the call and read by calls on any stream and of any thread.  So a call uses what it has built in its stream's
    order, and once its product is launched waits for the stream and only then shows the form to others (``_keep_form``): once in a form's life,
    where an event would have to be asked about on every call, and cannot be under capture.

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
        """The form ``name`` of the weight as it is now: the kept one, or a new one for ``_keep_form``.  One that is built while the stream is captured
        belongs to that graph, which writes it on every replay; with ``needed`` false, for a call that has another way, None in its place."""
        components = tuple(getattr(self, c) for c in self._FORM_COMPONENTS)
        kept, key = getattr(self, name), weight_key(components)
        if kept is not None and kept.key == key:
            return kept
        in_graph = capturing(components[0].device)
        if in_graph and not needed:
            return None
        into = kept.value if kept is not None and kept.key[::2] == key[::2] and not in_graph else None      # (the same tensors, written since)
        return WeightForm(self._build_form(name, into, *components), key, tuple(c.detach() for c in components))

    def _keep_form(self, name: str, form: WeightForm) -> None:
        """Keep a form that ``_weight_form`` gave, for calls on every stream."""
        kept = getattr(self, name)
        if form is kept or capturing(form.components[0].device):
            return
        if any(isinstance(getattr(type(self), c, None), property) for c in self._FORM_COMPONENTS):
            return                                            # (a parametrisation makes another tensor for every call)
        finish(form.components[0].device, every_stream=kept is not None)      # (calls on other streams may still read the one that goes)
        self.__dict__[name] = form

    def _drop_forms(self, moved_only: bool = False) -> None:
        """Forget the forms, or those whose components are not the layer's any more."""
        components = [getattr(self, c) for c in self._FORM_COMPONENTS]
        key = None if any(c is None for c in components) else weight_key(components)
        for name in self._FORMS:
            kept = getattr(self, name)
            if kept is not None and not (moved_only and kept.key == key):
                self.__dict__[name] = self.__dict__["_note"] = None

    def _load_from_state_dict(self, *args, **kwargs):
        super()._load_from_state_dict(*args, **kwargs)
        for name in self._FORMS:
            kept = getattr(self, name)
            if kept is not None and kept.key[::2] == weight_key([getattr(self, c) for c in self._FORM_COMPONENTS])[::2]:
                self._keep_form(name, self._weight_form(name))

    def __getstate__(self):
        return {**self.__dict__, **dict.fromkeys(self._FORMS), "_note": None}

    def __setstate__(self, state):
        super().__setstate__({**state, **dict.fromkeys(self._FORMS), "_note": None})         # (older pickles hold forms without a key)
