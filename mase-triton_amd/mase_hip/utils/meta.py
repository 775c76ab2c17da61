"""String/tuple normalisers used by the tensor-meta dataclasses
(same contract as src/mase_triton/utils/meta.py:4-25)."""
import torch


_NAMES: dict = {}      # names of the devices and dtypes seen (printing one costs more than looking it up)


def device_str(device) -> str:
    if isinstance(device, str):
        return device
    name = _NAMES.get(device)
    if name is None:
        name = _NAMES[device] = str(device)
    return name


def dtype_str(dtype) -> str:
    if isinstance(dtype, str):
        return dtype
    name = _NAMES.get(dtype)
    if name is None:
        name = _NAMES[dtype] = str(dtype).removeprefix("torch.")
    return name


def shape_tuple(shape) -> tuple:
    return tuple(shape) if isinstance(shape, torch.Size) else shape
