"""Projections to attention heads in one HIP pass: q/k norm, rotary embedding and ``[S, H*D] -> [H, S, D]``.

The processors' tensor operations for this (``svoo/models/wan/attention.py:153-215``,
``svoo/models/hunyuan10/attention.py:305-353, 536-575``) read and write Q and K about a dozen times; the HIP kernel
reads and writes each once, with the same roundings (the norm's result to bf16, fp32 products of the rotation, its
result to bf16).  :func:`qkv_heads` takes plain bf16 inference tensors only; for anything else - gradients, hooks,
tracing, transforms, autocast, other types or layouts - it returns None and the caller keeps its tensor operations.
"""

from __future__ import annotations

from typing import Optional, Tuple

import torch

from . import _lib

_GLOBAL_HOOKS = ("_global_forward_hooks", "_global_forward_pre_hooks", "_global_backward_hooks",
                 "_global_backward_pre_hooks")
_MODULE_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def plain_execution() -> bool:
    """No tracing, compilation, function transform, forward-mode level, dispatch or function mode, or autocast: a kernel
    launched on raw pointers then sees what the tensor operations would.  Some of these can only be asked of names that
    torch keeps to itself: where one is missing the answer is no."""
    try:
        return not (torch.jit.is_tracing() or torch.compiler.is_compiling()
                    or torch._C._functorch.peek_interpreter_stack() is not None
                    or torch.autograd.forward_ad._current_level >= 0
                    or torch._C._len_torch_dispatch_stack() > 0 or torch._C._len_torch_function_stack() > 0
                    or torch.is_autocast_enabled("cuda"))
    except (AttributeError, TypeError):
        return False


def _plain(t, dtype, device) -> bool:
    return (type(t) in (torch.Tensor, torch.nn.Parameter) and t.is_cuda and t.device == device and t.dtype == dtype
            and not (torch.is_grad_enabled() and t.requires_grad) and t.data_ptr() % 16 == 0)


def rms_norm_params(norm, width: int, device) -> Optional[tuple]:
    """``(weight or None, eps)`` when ``norm`` is exactly a ``torch.nn.RMSNorm`` over ``width`` elements whose call the
    kernel can stand in for (a bf16 weight, a given eps, no hooks or overridden forward), else None."""
    if type(norm) is not getattr(torch.nn, "RMSNorm", None) or norm.normalized_shape != (width,) or norm.eps is None:
        return None
    mod = torch.nn.modules.module
    if "forward" in norm.__dict__ or any(getattr(mod, n, None) for n in _GLOBAL_HOOKS) or \
            any(getattr(norm, n, None) for n in _MODULE_HOOKS):
        return None
    w = norm.weight
    if w is not None and not (_plain(w, torch.bfloat16, device) and w.is_contiguous()):
        return None
    return w, float(norm.eps)


def rows_ok(x, heads: int) -> bool:
    """``x [1, S, H*D]`` as rows the kernel reads: bf16, contiguous within a row, rows at 16-byte addresses, on the current
    device (a launch goes to that one, also on another's null stream)."""
    if type(x) not in (torch.Tensor, torch.nn.Parameter) or x.dim() != 3 or not x.is_cuda or \
            x.device.index != torch.cuda.current_device():
        return False
    b, s, dim = x.shape
    return (b == 1 and s > 0 and heads > 0 and dim in (64 * heads, 128 * heads) and dim <= 8192
            and _plain(x, torch.bfloat16, x.device) and x.stride(2) == 1 and x.stride(1) % 8 == 0)


def linear_ok(module, x, width: int) -> bool:
    """``module(x)`` is a plain projection whose result :func:`rows_ok` will take: a ``torch.nn.Linear`` to ``width``
    in bf16 without gradients or hooks, of ``x [1, T, C]``."""
    if type(module) is not torch.nn.Linear or module.out_features != width or "forward" in module.__dict__ or \
            any(getattr(torch.nn.modules.module, n, None) for n in _GLOBAL_HOOKS) or \
            any(getattr(module, n, None) for n in _MODULE_HOOKS):
        return False
    return (type(x) is torch.Tensor and x.dim() == 3 and x.shape[0] == 1 and x.is_cuda
            and all(_plain(t, torch.bfloat16, x.device) for t in (x, module.weight, module.bias) if t is not None))


def tables_ok(tables, shape, device) -> bool:
    """Rotary ``(cos, sin)`` as contiguous fp32 tensors of ``shape`` on ``device``."""
    return len(tables) == 2 and all(isinstance(t, torch.Tensor) and tuple(t.shape) == tuple(shape)
                                    and _plain(t, torch.float32, device) and t.is_contiguous() for t in tables)


def qkv_heads(q, k, v, heads: int, *, norm: int = 0, q_norm=(None, 0.0), k_norm=(None, 0.0), rope=None,
              rope_rows: int = 0, per_element: bool = False, out=None, out_row0: int = 0) -> Tuple[torch.Tensor, ...]:
    """``q, k, v [1, S, H*D]`` (checked by :func:`rows_ok`) -> three ``[1, H, S, D]`` tensors.

    ``norm``: 0 none, 1 RMSNorm of q and k over the whole row, 2 per head, with ``(weight, eps)`` each; ``rope``: fp32
    ``(cos, sin)`` of ``rope_rows`` rows of D, applied to the first ``rope_rows`` rows of q and k on interleaved pairs:
    both elements of a pair by its even cosine and odd sine (Wan), or with ``per_element`` each by its own (HunyuanVideo).
    ``out``: three ``[1, H, R, D]`` tensors to fill from row ``out_row0`` instead of new ones of S rows."""
    _, s, dim = q.shape
    d = dim // heads
    if out is None:
        out = tuple(torch.empty(1, heads, s, d, dtype=q.dtype, device=q.device) for _ in range(3))
    cos, sin = rope if rope is not None else (None, None)
    _lib.call("svoo_qkv_heads", q.data_ptr(), k.data_ptr(), v.data_ptr(), q.stride(1), k.stride(1), v.stride(1),
              out[0].data_ptr(), out[1].data_ptr(), out[2].data_ptr(), s, heads, d, out[0].shape[2], out_row0, norm,
              _lib.ptr(q_norm[0]), _lib.ptr(k_norm[0]), q_norm[1], k_norm[1], _lib.ptr(cos), _lib.ptr(sin), rope_rows,
              int(per_element), _lib.stream_of(q.device))
    return out
