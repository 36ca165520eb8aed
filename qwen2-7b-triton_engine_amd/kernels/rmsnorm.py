"""RMSNorm on a hand-written gfx950 kernel (``awq_fp16_rmsnorm``).

``model/qwen2.py:15-22`` in one launch: ``x * rsqrt(mean(x^2) + eps) * w`` in
fp32, rounded once to fp16.
"""
from __future__ import annotations

import torch

from . import _native
from .awq_gemm import _OnDevice, _aligned16, _stream_handle

__all__ = ["rmsnorm", "MAX_H"]

MAX_H = 16384   # the longest row the kernel holds in registers


def rmsnorm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """fp16 ``[..., H]`` from fp16 ``x [..., H]`` and ``w [H]``; H a multiple of 8, at
    most ``MAX_H``."""
    H = x.shape[-1]
    if x.dtype != torch.float16 or w.dtype != torch.float16 or tuple(w.shape) != (H,):
        raise ValueError(f"x and w must be fp16, w of shape {(H,)}, got {x.dtype}, {w.dtype} {tuple(w.shape)}")
    if H % 8 != 0 or not 0 < H <= MAX_H:
        raise ValueError(f"H = {H} must be a multiple of 8 and at most {MAX_H}")
    if x.device.type != "cuda" or w.device != x.device:
        raise ValueError(f"x and w must be on one ROCm device, got {x.device} and {w.device}")
    x, w = _aligned16(x.contiguous()), _aligned16(w.contiguous())
    out = torch.empty_like(x)
    with _OnDevice(x.device):
        st = _native.lib().awq_fp16_rmsnorm(x.data_ptr(), w.data_ptr(), out.data_ptr(), x.numel() // H, H, eps,
                                            _stream_handle(x.device))
    _native.check(st, "awq_fp16_rmsnorm")
    return out
