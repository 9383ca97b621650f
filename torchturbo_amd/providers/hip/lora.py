"""HIP LoRA residual of a grouped linear layer (``GroupedMLPLoRA``).

``lora_residual(base, x, a, b, counts, scaling)`` is
``base + grouped_matmul(grouped_matmul(x.to(a.dtype), a), b).to(base.dtype) * scaling``
(``engine/peft/lora.py:640-725``) with the same roundings, without the fp32
copy of ``x`` and the fp32 product behind it; ``supported`` says which operands
it takes (16-bit rows, fp32 adapters of rank 64 or less, 16-byte aligned).
"""

from __future__ import annotations

import torch

from ... import _lib as L
from ...dispatch import OpImpl, OpImplKind, register_op
from ...runtime import TurboDevice
from . import PRIORITY
from ._functions import device_counts, require_cuda
from .available import hip_available

MAX_RANK = 64


class LoRAResidual(torch.autograd.Function):
    """``(base, x, a, b, counts, scaling) -> y``; the gradient of ``base`` is
    the output's."""

    @staticmethod
    def forward(ctx, base, x, a, b, counts, scaling):
        base, x, a, b = (v.contiguous() for v in (base, x, a, b))
        E, K, r = a.shape
        M, N = base.shape
        dev, code = x.device, L.dtype_code(x.dtype)
        h = torch.empty((M, r), dtype=torch.float32, device=dev)
        y = torch.empty_like(base)
        st = L.stream(dev)
        L.call("tt_lora_down", L.ptr(x), L.ptr(a), code, M, K, r, 0, 1.0, E, L.ptr(counts),
               L.ptr(h), st)
        L.call("tt_lora_up", L.ptr(h), L.ptr(b), L.ptr(base), code, M, N, r, 0, scaling, E,
               L.ptr(counts), L.ptr(y), st)
        ctx.save_for_backward(x, a, b, h, counts)
        ctx.scaling = scaling
        return y

    @staticmethod
    def backward(ctx, dy):
        x, a, b, h, counts = ctx.saved_tensors
        s = ctx.scaling
        need = ctx.needs_input_grad
        E, K, r = a.shape
        g = dy.to(x.dtype).contiguous()
        if not aligned(g):
            g = g.clone()
        M, N = g.shape
        dev, code = x.device, L.dtype_code(x.dtype)
        st = L.stream(dev)
        dx = da = db = None
        if need[1] or need[2]:
            dh = torch.empty_like(h)
            L.call("tt_lora_down", L.ptr(g), L.ptr(b), code, M, N, r, 1, s, E, L.ptr(counts),
                   L.ptr(dh), st)
        if need[3]:
            db = torch.empty_like(b)
            L.call("tt_lora_wgrad", L.ptr(g), L.ptr(h), code, M, N, r, 1, s, E, L.ptr(counts),
                   L.ptr(db), st)
        if need[1]:
            dx = torch.empty_like(x)
            L.call("tt_lora_up", L.ptr(dh), L.ptr(a), None, code, M, K, r, 1, 1.0, E,
                   L.ptr(counts), L.ptr(dx), st)
        if need[2]:
            da = torch.empty_like(a)
            L.call("tt_lora_wgrad", L.ptr(x), L.ptr(dh), code, M, K, r, 0, 1.0, E, L.ptr(counts),
                   L.ptr(da), st)
        return dy if need[0] else None, dx, da, db, None, None


def aligned(t) -> bool:
    """Whether the kernels can read ``t``: a tensor that is not contiguous is copied first."""
    return t.data_ptr() % 16 == 0 or not t.is_contiguous()


def supported(base, x, a, b) -> bool:
    r = a.shape[-1]
    return (base.is_cuda and x.dtype in (torch.bfloat16, torch.float16) and base.dtype == x.dtype
            and base.dim() == 2 and x.dim() == 2 and a.dtype == b.dtype == torch.float32
            and 1 <= r <= MAX_RANK and x.shape[1] % 8 == 0 and base.shape[1] % 8 == 0
            and x.shape[0] == base.shape[0] and a.shape[1] == x.shape[1]
            and b.shape[1:] == (r, base.shape[1]) and a.shape[0] == b.shape[0]
            and all(aligned(t) for t in (base, x, a, b)))


@register_op(op_name="lora_residual", impl_name="hip_lora_residual", kind=OpImplKind.CUSTOM,
             priority=PRIORITY, devices=(TurboDevice.CUDA,))
class HipLoRAResidual(OpImpl):
    def available(self) -> bool:
        return hip_available()

    def __call__(self, base, x, a, b, counts, scaling):
        """None for operands that ``supported`` leaves to the composition."""
        if not supported(base, x, a, b):
            return None
        dev = require_cuda(base, x, a, b)
        counts = device_counts(counts, a.shape[0], dev, m=x.shape[0])
        return LoRAResidual.apply(base, x, a, b, counts, float(scaling))
