"""The engine's attention on hand-written gfx950 kernels.

``attention_decode`` is one new position over a static KV cache, from the
fused QKV projection to the attention output: RoPE, the cache's new row,
softmax(q K^T / sqrt(d)) V (``model/qwen2.py:104-163``,
``kernels/rope.py:41-57``) -- two launches.  ``attention_prefill`` is the same
for a prompt's positions 0 .. S - 1.  q after RoPE and the probabilities are
fp32 values that enter the matrix cores as sums of two fp16 values (23 bits);
scores, softmax and sums are fp32.
"""
from __future__ import annotations

import torch

from . import _native
from .awq_gemm import _OnDevice, _stream_handle

__all__ = ["attention_decode", "attention_prefill", "attention_served"]


def attention_served(num_heads: int, num_kv_heads: int, head_dim: int, max_seq: int) -> bool:
    """Whether the kernels serve these head counts, head size and cache length."""
    return _native.lib().awq_fp16_attention_decode_workspace(num_heads, num_kv_heads, head_dim, max_seq) > 0


def _check_cache(dev, k_cache, v_cache, cos, sin):
    """(kv heads, cache length, head size) of one layer's caches."""
    if k_cache.dim() != 3 or k_cache.shape != v_cache.shape:
        raise ValueError(f"k_cache {tuple(k_cache.shape)} and v_cache {tuple(v_cache.shape)} must be equal 3-D shapes")
    kvh, max_seq, hd = k_cache.shape
    for t, what, dtype, shape in ((k_cache, "k_cache", torch.float16, (kvh, max_seq, hd)),
                                  (v_cache, "v_cache", torch.float16, (kvh, max_seq, hd)),
                                  (cos, "cos", torch.float32, (max_seq, hd)),
                                  (sin, "sin", torch.float32, (max_seq, hd))):
        if t.dtype != dtype or tuple(t.shape) != shape or not t.is_contiguous() or t.device != dev:
            raise ValueError(f"{what} must be a contiguous {dtype} tensor {shape} on {dev}")
    return kvh, max_seq, hd


def attention_decode(qkv: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cos: torch.Tensor,
                     sin: torch.Tensor, pos: torch.Tensor, num_heads: int) -> torch.Tensor:
    """Attention output fp16 ``[1, num_heads * head_dim]`` of the position
    ``pos`` (int64 ``[1]``, on the device); its k and v go into row ``pos`` of
    ``k_cache`` / ``v_cache`` ``[kv_heads, max_seq, head_dim]``.  The host does not
    read the position: outside the cache the caches stay as they are and the
    output is NaN."""
    dev = qkv.device
    kvh, max_seq, hd = _check_cache(dev, k_cache, v_cache, cos, sin)
    if qkv.dtype != torch.float16 or qkv.numel() != (num_heads + 2 * kvh) * hd or not qkv.is_contiguous():
        raise ValueError(f"qkv must be a contiguous fp16 tensor of {(num_heads + 2 * kvh) * hd} values")
    if pos.dtype != torch.int64 or pos.numel() != 1 or pos.device != dev:
        raise ValueError(f"pos must be an int64 [1] tensor on {dev}")
    L = _native.lib()
    ws = torch.empty(L.awq_fp16_attention_decode_workspace(num_heads, kvh, hd, max_seq), dtype=torch.uint8, device=dev)
    out = torch.empty((1, num_heads * hd), dtype=torch.float16, device=dev)
    with _OnDevice(dev):
        st = L.awq_fp16_attention_decode(qkv.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(),
                                         sin.data_ptr(), pos.data_ptr(), out.data_ptr(), num_heads, kvh, hd, max_seq,
                                         ws.data_ptr(), ws.numel(), _stream_handle(dev))
    _native.check(st, "awq_fp16_attention_decode")
    return out


def attention_prefill(qkv: torch.Tensor, k_cache: torch.Tensor, v_cache: torch.Tensor, cos: torch.Tensor,
                      sin: torch.Tensor, num_heads: int) -> torch.Tensor:
    """Causal attention fp16 ``[S, num_heads * head_dim]`` of positions 0 .. S - 1
    (``qkv`` fp16 ``[S, (num_heads + 2 kv_heads) * head_dim]``); their k and v go
    into the first S rows of the caches."""
    dev = qkv.device
    kvh, max_seq, hd = _check_cache(dev, k_cache, v_cache, cos, sin)
    if qkv.dtype != torch.float16 or qkv.dim() != 2 or qkv.shape[1] != (num_heads + 2 * kvh) * hd \
            or not qkv.is_contiguous():
        raise ValueError(f"qkv must be a contiguous fp16 tensor [S, {(num_heads + 2 * kvh) * hd}]")
    S = qkv.shape[0]
    if S > max_seq:
        raise ValueError(f"{S} positions exceed the cache's {max_seq}")
    L = _native.lib()
    ws = torch.empty(L.awq_fp16_attention_prefill_workspace(S, kvh, hd), dtype=torch.uint8, device=dev)
    out = torch.empty((S, num_heads * hd), dtype=torch.float16, device=dev)
    with _OnDevice(dev):
        st = L.awq_fp16_attention_prefill(qkv.data_ptr(), k_cache.data_ptr(), v_cache.data_ptr(), cos.data_ptr(),
                                          sin.data_ptr(), out.data_ptr(), S, num_heads, kvh, hd, max_seq,
                                          ws.data_ptr(), ws.numel(), _stream_handle(dev))
    _native.check(st, "awq_fp16_attention_prefill")
    return out
