"""HIP blockwise FP8 quantisation (``Fp8GroupedMLP.requantize``).

``quantize_fp8_blocks(weight, q, scale)`` writes the e4m3 codes and 128x128
block scales of a weight in one pass over it, the bytes that the torch
composition in ``Fp8GroupedMLP.requantize`` gives (the inverse of
``scripts/dequant/bailing.py:57-102``), and returns True. Operands the kernel
does not cover (weights that are not bf16, tensors that are not contiguous or
not all on the weight's GPU) return False and are left to the caller.
"""

from __future__ import annotations

import torch
from torch.autograd.graph import increment_version

from ... import _lib as L
from ...dispatch import OpImpl, OpImplKind, register_op
from ...runtime import TurboDevice
from . import PRIORITY
from .available import hip_available


@register_op(op_name="quantize_fp8_blocks", impl_name="hip_quantize_fp8_blocks",
             kind=OpImplKind.CUSTOM, priority=PRIORITY, devices=(TurboDevice.CUDA,))
class HipQuantizeFp8Blocks(OpImpl):
    def available(self) -> bool:
        return hip_available()

    def __call__(self, weight, q, scale) -> bool:
        if not (weight.is_cuda and q.device == weight.device == scale.device):
            return False
        if (weight.dtype != torch.bfloat16 or q.dtype != torch.float8_e4m3fn
                or scale.dtype not in (torch.bfloat16, torch.float32)
                or not (weight.is_contiguous() and q.is_contiguous() and scale.is_contiguous())
                or weight.data_ptr() % 16 or q.data_ptr() % 8):
            return False
        E, R, C = weight.shape
        if (R % 128 or C % 128 or q.shape != weight.shape
                or scale.shape != (E, R // 128, C // 128)):
            return False
        L.call("tt_fp8_quantize_blocks", L.ptr(weight), L.dtype_code(weight.dtype), E, R, C,
               L.ptr(q), L.ptr(scale), L.dtype_code(scale.dtype), L.stream(weight.device))
        # Written in place: a backward that saved the old values must see it.
        increment_version(q)
        increment_version(scale)
        return True
