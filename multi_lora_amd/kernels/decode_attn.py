"""The decoder's decode attention and SiLU gate as single HIP launches.

``decode_attention`` covers what ``decoder.Attention`` does for one new token
per sequence over a ``StaticKV`` layer; ``silu_mul`` its MLP's gate.  Both
return None (nothing launched) for calls they do not take: other dtypes,
devices and layouts, and calls whose operations torch has to see (autograd in
either mode, tracing and compilation, function transforms, dispatch and
function modes); the caller then runs the torch operations.
"""

from __future__ import annotations

from typing import Optional

import torch
from torch.autograd import forward_ad
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

from .. import _ffi

_DTYPES = (torch.float16, torch.bfloat16)
# Longest cache taken.  One workgroup takes a key head's whole cache: with
# fewer than 64 of them the chip is nearly idle, and past 1024 positions torch's
# launches catch up (4 key heads, 2048 positions: 53.0 against 51.8 us; 64: 64.3
# against 64.5; at 512 key heads 166 against 204, and at 520 positions 57 against
# 96).  Eight query heads a key head fill a CU's LDS with one workgroup, and
# torch's catch up earlier (the layer with its projections, 1 key head, 1024
# positions: 60-62 against 52-53; 4: 79 against 75; 128 key heads, 2048 positions:
# 114-118 against 110-111, 1024: faster).
FEW_HEADS = 64


def _max_len(key_heads: int, rep: int) -> int:
    if rep == 8:
        return 1024 if key_heads >= FEW_HEADS else 600
    return 2048 if key_heads >= FEW_HEADS else 1024


def _followed() -> bool:
    """Whether something follows the torch operations run now: a launch past
    torch would drop out of it (a forward-mode tangent, a recorded graph, a
    batched dimension), although its tensors look plain."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or forward_ad._current_level >= 0
            or torch._C._functorch.peek_interpreter_stack() is not None
            or torch._C._len_torch_dispatch_stack() > 0
            or (torch._C._len_torch_function_stack() > 0
                and any(type(m) is not DeviceContext for m in _get_current_function_mode_stack())))


def _plain(*tensors: torch.Tensor) -> bool:
    if _followed():
        return False
    first = tensors[0]
    # A launch goes to the current device; torch's operations follow the tensor.
    return (first.is_cuda and first.dtype in _DTYPES and first.device.index == torch.cuda.current_device()
            and all(type(t) is torch.Tensor and t.device == first.device for t in tensors)
            and not (torch.is_grad_enabled() and any(t.requires_grad for t in tensors)))


def decode_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor,
                     keys: torch.Tensor, values: torch.Tensor, hide: torch.Tensor, pos: torch.Tensor,
                     scale: float) -> Optional[torch.Tensor]:
    """Rotary on ``q [b, heads*d]`` and ``k [b, kv_heads*d]``, the new key and
    value into ``keys [b, kv_heads, d, L]`` / ``values [b, kv_heads, L, d]`` at
    ``pos`` (one int64 on the device), and the attention of every row over the
    cache, except the positions ``hide [b, 1, 1, L]`` marks; ``[b, heads*d]``.
    A ``pos`` outside the cache, which only the device knows, writes nothing
    and makes the result NaN."""
    if values.dim() != 4:
        return None
    b, kv_heads, length, d = values.shape
    if d not in (64, 128) or q.dim() != 2 or q.shape[1] % d or b == 0:
        return None
    heads = q.shape[1] // d
    if heads % kv_heads or heads // kv_heads not in (1, 2, 4, 8) or length > _max_len(b * kv_heads, heads // kv_heads):
        return None
    if not _plain(q, k, v, cos, sin, keys, values, hide, pos):
        return None
    rows = (q, k, v)
    if any(t.dtype != q.dtype for t in (k, v, cos, sin, keys, values)) or any(t.stride(1) != 1 for t in rows):
        return None
    if q.shape[0] != b or any(t.shape != (b, kv_heads * d) for t in (k, v)):
        return None
    if keys.shape != (b, kv_heads, d, length) or not keys.is_contiguous() or not values.is_contiguous():
        return None
    if cos.shape != (b, 1, d) or sin.shape != (b, 1, d) or cos.stride() != sin.stride() or cos.stride(2) != 1:
        return None
    if hide.dtype != torch.bool or hide.shape != (b, 1, 1, length) or hide.stride(3) != 1:
        return None
    if pos.dtype != torch.int64 or pos.numel() != 1 or values.data_ptr() % 16:
        return None
    if (keys.is_inference() or values.is_inference()) and not torch.is_inference_mode_enabled():
        return None  # torch refuses the write
    out = torch.empty((b, heads * d), dtype=q.dtype, device=q.device)
    rc = _ffi.lib().mlora_decode_attention(
        q.data_ptr(), q.stride(0), k.data_ptr(), k.stride(0), v.data_ptr(), v.stride(0), cos.data_ptr(), sin.data_ptr(),
        cos.stride(0), keys.data_ptr(), values.data_ptr(), hide.data_ptr(), hide.stride(0), pos.data_ptr(),
        out.data_ptr(), heads * d, b, heads, kv_heads, d, length, float(scale), _ffi.dtype_code(q.dtype),
        _ffi.stream_ptr(q.device))
    if rc == -2:
        return None
    _ffi.check(rc, "mlora_decode_attention")
    # Written in place: a backward pass that saved the caches must notice.
    torch.autograd.graph.increment_version((keys, values))
    return out


def silu_mul(gate: torch.Tensor, up: torch.Tensor) -> Optional[torch.Tensor]:
    """``silu(gate) * up`` of two tensors of one shape and row stride (the
    halves of a fused gate|up output)."""
    if not _plain(gate, up) or gate.dtype != up.dtype or gate.shape != up.shape or gate.dim() < 2:
        return None
    width = gate.shape[-1]
    if gate.numel() == 0 or gate.stride() != up.stride() or gate.stride(-1) != 1 or width % 8:
        return None
    stride, rows = gate.stride(-2), gate.numel() // width
    span = stride
    for n, st in zip(reversed(gate.shape[:-1]), reversed(gate.stride()[:-1])):  # rows equally spaced
        if n != 1 and st != span:
            return None
        span *= n
    if stride % 8 or stride < width or (gate.data_ptr() | up.data_ptr()) % 16:
        return None
    out = torch.empty(gate.shape, dtype=gate.dtype, device=gate.device)
    rc = _ffi.lib().mlora_silu_mul(gate.data_ptr(), up.data_ptr(), stride, out.data_ptr(), rows, width,
                                   _ffi.dtype_code(gate.dtype), _ffi.stream_ptr(gate.device))
    if rc == -2:
        return None
    _ffi.check(rc, "mlora_silu_mul")
    return out
