"""Helpers shared by the op modules: env flags, dtype checks, shape rules."""

from __future__ import annotations

import os

import torch
from torch.autograd import forward_ad

ACT_DTYPES = (torch.float16, torch.bfloat16)
FLOAT_DTYPES = (torch.float16, torch.bfloat16, torch.float32, torch.float64)


def ci_safe_mode_enabled() -> bool:
    """MLX_METAL_CI_SAFE_MODE=1 routes ops to their ``reference_*`` path, as in
    the reference (ops/quant_ops.py:33-34).  It is an explicit opt-in for hosts
    without a GPU; it is never set implicitly."""
    return os.environ.get("MLX_METAL_CI_SAFE_MODE", "0") == "1"


def env_flag(name: str) -> bool:
    return os.environ.get(name, "0") == "1"


def finfo_max(dtype: torch.dtype) -> float:
    return float(torch.finfo(dtype).max)


def scales_for_kernel(scales: torch.Tensor, zeros: torch.Tensor | None):
    """fp16 scales/zeros go to the kernels as they are; any other float dtype
    is promoted to fp32 (the reference promotes everything to fp32 at the
    kernel boundary, ops/quant_ops.py:424)."""
    use_f16 = scales.dtype == torch.float16 and (zeros is None or zeros.dtype == torch.float16)
    target = torch.float16 if use_f16 else torch.float32
    return as_dense(scales, target), as_dense(zeros, target)


def as_dense(t, dtype):
    """``t`` contiguous and in ``dtype`` (itself when it is; None stays None)."""
    if t is None or (t.dtype == dtype and t.is_contiguous()):
        return t
    return t.to(dtype).contiguous()


def values_only(*tensors: torch.Tensor) -> bool:
    """Whether a kernel that reads the tensors' memory does all that tensor ops
    would: no gradient to record, no forward-mode tangent, no function transform
    (vmap, jvp, grad), no tracing, dispatch mode or tensor subclass."""
    if (torch.compiler.is_compiling() or torch._C._is_tracing() or torch._C._len_torch_dispatch_stack()
            or torch._C._functorch.peek_interpreter_stack() is not None):  # (there even new tensors are wrapped)
        return False
    grad, dual = torch.is_grad_enabled(), forward_ad._current_level >= 0
    for t in tensors:
        if type(t) is not torch.Tensor and type(t) is not torch.nn.Parameter:
            return False
        if (grad and t.requires_grad) or (dual and forward_ad.unpack_dual(t).tangent is not None):
            return False
    return True


def as_u8(t: torch.Tensor) -> torch.Tensor:
    return (t if t.dtype == torch.uint8 else t.to(torch.uint8)).contiguous()
