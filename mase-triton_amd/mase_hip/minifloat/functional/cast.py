"""Public minifloat casts (API of src/mase_triton/minifloat/functional/cast.py:10-90)."""
from __future__ import annotations

import torch
from torch import Tensor

from ...utils.meta import device_str, dtype_str, shape_tuple
from ... import _lib
from ...dtype import TORCH_DTYPE_TO_CODE
from .. import kernels
from ..meta import MinifloatMeta, MinifloatTensorMeta


def extract_minifloat_component(tensor: Tensor, minifloat_meta: MinifloatMeta) -> tuple[Tensor, MinifloatTensorMeta]:
    """Quantise ``tensor``: returns ``(uint16 codes, tensor_meta)``.

    The reference widens to float32 before its kernel (:27); the HIP kernel reads float16 and
    bfloat16 directly, which yields the same codes with half the read traffic.
    """
    tensor_meta = MinifloatTensorMeta(
        device=device_str(tensor.device), dtype=dtype_str(tensor.dtype), shape=shape_tuple(tensor.shape),
        meta=minifloat_meta)
    codes = _lib.host().minifloat(0, tensor, minifloat_meta._codes, None)
    return kernels.extract_minifloat_component(tensor, minifloat_meta) if codes is None else codes, tensor_meta


def compose_minifloat_component(element: Tensor, tensor_meta: MinifloatTensorMeta,
                                output_dtype: torch.dtype | None = None) -> Tensor:
    """Dequantise codes; ``output_dtype`` defaults to the dtype recorded at extraction."""
    if output_dtype is None:
        output_dtype = getattr(torch, tensor_meta.dtype)
    out = _lib.host().minifloat(1, element, tensor_meta.meta._codes, TORCH_DTYPE_TO_CODE.get(output_dtype, -1))
    return kernels.compose_minifloat_component(element, tensor_meta.meta, output_dtype=output_dtype) if out is None else out


def quantize_dequantize(tensor: Tensor, minifloat_meta: MinifloatMeta, output_dtype: torch.dtype | None = None) -> Tensor:
    """Round ``tensor`` to the minifloat grid (fused single-pass kernel)."""
    out = _lib.host().minifloat(2, tensor, minifloat_meta._codes, None if output_dtype is None else TORCH_DTYPE_TO_CODE.get(output_dtype, -1))
    if out is not None:
        return out
    return kernels.quantize_dequantize(tensor, minifloat_meta, tensor.dtype if output_dtype is None else output_dtype)
