"""The element-wise steps between a layer's matrix products on the fused HIP kernels
(``csrc/layer_ops.hip``), each beside the torch ops it replaces.

The kernels run where nothing else can be watching the tensors in between: grad mode off, plain
tensors of the current device and of one dtype, no autocast, tracing, functorch transform, forward-mode AD or
dispatch / function mode, and sub-modules of exactly the expected class without hooks or replaced
methods.  Everything else takes the torch ops.
"""
from __future__ import annotations

import ctypes
from typing import Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import module as _module

from . import _lib
from .hip_kernels import on_current_device, rms_default_eps, unobserved

_DTYPES = (torch.bfloat16, torch.float16, torch.float32)


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def fusable(x: torch.Tensor) -> bool:
    """Whether kernels outside torch's dispatcher may take this tensor's place in the op sequence."""
    return (type(x) is torch.Tensor and on_current_device(x) and x.dtype in _DTYPES
            and not torch.is_grad_enabled()
            and not torch.is_autocast_enabled("cuda") and unobserved())


def plain(m, cls) -> bool:
    """A module of exactly ``cls`` whose call does no more than its own ``forward``."""
    return (type(m) is cls and not m._forward_hooks and not m._forward_pre_hooks
            and not m._backward_hooks and not m._backward_pre_hooks
            and "forward" not in m.__dict__ and m._compiled_call_impl is None
            and not _module._has_any_global_hook())


def _rows(*ts) -> bool:
    """Contiguous 16-byte aligned tensors (None: absent)."""
    return all(t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0) for t in ts)


_PLAIN = (torch.Tensor, nn.Parameter)


def _parameter_ok(p, shape: tuple, x: torch.Tensor) -> bool:
    """A plain tensor of exactly ``shape`` beside ``x``, in its type: what torch's op would refuse or
    convert must reach that op."""
    return type(p) in _PLAIN and tuple(p.shape) == shape and p.dtype == x.dtype and p.device == x.device


def _row_fits(d: int, dtype: torch.dtype) -> bool:
    n = 16 // dtype.itemsize
    return d % n == 0 and d <= 1024 * n


def _few_rows(x: torch.Tensor, n: int, k: int) -> bool:
    """Whether ``csrc/rows_linear.hip`` takes x [M, k] times [n, k]: M <= 16, x up to 32 KB, a row up
    to 4 KB, the weight up to 16 MB.  The library spends 19.5 us of host time on such a product, the
    kernel's call 11; on the device, in us, kernel / library: bf16 n3328 k1024 M1 2.9 / 4.5, M16
    3.7 / 4.6; fp32 there M1 4.4 / 5.4, M16 5.6 / 5.6; bf16 n1536 k2048 M4 4.3 / 5.1,
    M16 5.3 / 5.1; past the lines bf16 n6400 k2048 M1 6.5 / 5.9, n16384 k4096 M16 30 / 22."""
    size = x.dtype.itemsize
    return (0 < x.numel() <= 16 * k and x.numel() * size <= 32768 and k * size <= 4096 and 0 < n
            and n * k * size <= 2 ** 24 and k * size % 16 == 0)


def rows_linear(x: torch.Tensor, weight: torch.Tensor) -> torch.Tensor:
    """``F.linear(x, weight)`` of a decode step, x [B, 1, hidden]: a few rows on
    ``csrc/rows_linear.hip``, more on the library."""
    n, k = weight.shape
    if (x.shape[-1] == k and _few_rows(x, n, k) and fusable(x)
            and type(weight) in (torch.Tensor, nn.Parameter) and weight.dtype == x.dtype
            and weight.device == x.device and _rows(x, weight)):
        out = torch.empty((*x.shape[:-1], n), device=x.device, dtype=x.dtype)
        _lib.check(_lib.load().vmi_rows_linear(_ptr(x), k, _ptr(weight), _lib.dtype_code(x.dtype), _ptr(out),
                                               x.numel() // k, n, k, _lib.stream_handle(x.device)),
                   "vmi_rows_linear")
        return out
    return F.linear(x, weight)


def rows_call(linear, x: torch.Tensor) -> torch.Tensor:
    """``linear(x)`` for a projection without bias, as :func:`rows_linear` where that is the same."""
    if plain(linear, nn.Linear) and linear.bias is None:
        return rows_linear(x, linear.weight)
    return linear(x)


def _norm_ok(norm, x: torch.Tensor) -> bool:
    d = x.shape[-1]
    return norm is None or (plain(norm, nn.RMSNorm) and tuple(norm.normalized_shape) == (d,)
                            and _parameter_ok(norm.weight, (d,), x) and _rows(norm.weight))


def _eps(norm, dtype) -> float:
    if norm is None:
        return 0.0
    return rms_default_eps(dtype) if norm.eps is None else float(norm.eps)


def norm_add(a: torch.Tensor, norm1=None, c: Optional[torch.Tensor] = None,
             b: Optional[torch.Tensor] = None, norm2=None) -> Tuple[torch.Tensor, Optional[torch.Tensor]]:
    """``s = b + (c + norm1(a))`` (absent terms left out) and ``norm2(s)``: (s, norm2(s) or None)."""
    d = a.shape[-1]
    same = all(t is None or (type(t) is torch.Tensor and t.dtype == a.dtype and t.shape == a.shape
                             and t.device == a.device) for t in (b, c))
    if (fusable(a) and same and a.numel() > 0 and _row_fits(d, a.dtype) and _rows(a, b, c)
            and _norm_ok(norm1, a) and _norm_ok(norm2, a)):
        s = torch.empty_like(a)
        out = None if norm2 is None else torch.empty_like(a)
        _lib.check(_lib.load().vmi_norm_add(
            _ptr(a), _ptr(None if norm1 is None else norm1.weight), _eps(norm1, a.dtype), _ptr(c),
            _ptr(b), _ptr(s), _ptr(None if norm2 is None else norm2.weight), _eps(norm2, a.dtype),
            _ptr(out), _lib.dtype_code(a.dtype), a.numel() // d, d, _lib.stream_handle(a.device)),
            "vmi_norm_add")
        return s, out
    s = a if norm1 is None else norm1(a)
    if c is not None:
        s = c + s
    if b is not None:
        s = b + s
    return s, None if norm2 is None else norm2(s)


def situ_glu(g: torch.Tensor, u: torch.Tensor, beta1: float, beta2: float) -> torch.Tensor:
    """``[b1 tanh(g / b1) sigmoid(g)] * [b2 tanh(u / b2)]``."""
    if (fusable(g) and isinstance(beta1, (int, float)) and isinstance(beta2, (int, float))
            and type(u) in _PLAIN and u.dtype == g.dtype and u.device == g.device and u.shape == g.shape
            and g.numel() > 0 and g.numel() % (16 // g.dtype.itemsize) == 0 and _rows(g, u)):
        out = torch.empty_like(g)
        _lib.check(_lib.load().vmi_situ_glu(_ptr(g), _ptr(u), _lib.dtype_code(g.dtype), beta1, beta2,
                                            _ptr(out), g.numel(), _lib.stream_handle(g.device)),
                   "vmi_situ_glu")
        return out
    return (beta1 * torch.tanh(g / beta1) * torch.sigmoid(g)) * (beta2 * torch.tanh(u / beta2))


def mcmoe_coef(logits: torch.Tensor, sig: torch.Tensor, vproj: torch.Tensor, top_k: int,
               components: Optional[int] = None) -> torch.Tensor:
    """``vproj * sigmoid(sig) * weight`` [n, C * r] of C = ``components`` (by default as many as
    logits), with the weights the softmax over the top-k logits (keep-top-k before the softmax,
    mcmoe.py:82-87), 0 off the top k."""
    n = logits.shape[0]
    C = logits.shape[1] if components is None else components
    r = vproj.shape[1] // C
    if (fusable(logits) and all(type(t) in _PLAIN and t.dtype == logits.dtype and t.device == logits.device
                                and tuple(t.shape) == (n, C * r) for t in (sig, vproj))
            and tuple(logits.shape) == (n, C) and n > 0 and 1 <= top_k <= C <= 64 and 0 < r <= 4096
            and r % (16 // logits.dtype.itemsize) == 0 and _rows(sig, vproj) and logits.is_contiguous()):
        coef = torch.empty_like(vproj)
        _lib.check(_lib.load().vmi_mcmoe_coef(_ptr(logits), _ptr(sig), _ptr(vproj),
                                              _lib.dtype_code(logits.dtype), top_k, _ptr(coef), n, C, r,
                                              _lib.stream_handle(logits.device)), "vmi_mcmoe_coef")
        return coef
    top_l, top_i = torch.topk(logits, k=top_k, dim=-1)
    masked = torch.full_like(logits, float("-inf")).scatter(-1, top_i, top_l)
    weights = torch.softmax(masked, dim=-1)                   # exactly 0 off the top k
    return (vproj.view(n, C, r) * torch.sigmoid(sig).view(n, C, r) * weights.unsqueeze(-1)).reshape(n, C * r)


class HaltingState:
    """The adaptive-depth loop's accumulators on the fused update (``vmi_halting_update``);
    :meth:`start` gives None where the torch ops have to run."""

    def __init__(self, linear, threshold, final_h, acc, depth):
        self.linear, self.final_h, self.acc, self.depth = linear, final_h, acc, depth
        # the comparison of a tensor with a number takes the number in the tensor's type
        self.threshold = float(torch.tensor(threshold, dtype=acc.dtype))

    @staticmethod
    def start(linear, threshold, h, final_h, acc, depth) -> Optional["HaltingState"]:
        d = h.shape[-1]
        ok = (fusable(h) and plain(linear, nn.Linear) and isinstance(threshold, (int, float))
              and _parameter_ok(linear.weight, (1, d), h) and _parameter_ok(linear.bias, (1,), h)
              and h.numel() > 0 and _row_fits(d, h.dtype) and _rows(h, final_h, linear.weight))
        return HaltingState(linear, threshold, final_h, acc, depth) if ok else None

    def _run(self, out, h, h_next, active, still, mode: int) -> None:
        _lib.check(_lib.load().vmi_halting_update(
            _ptr(out), _ptr(h), _ptr(h_next), _ptr(self.linear.weight), _ptr(self.linear.bias),
            _ptr(self.acc), _ptr(self.depth), _ptr(active), _ptr(still), _ptr(self.final_h),
            self.threshold, mode, _lib.dtype_code(h.dtype), h.numel() // h.shape[-1], h.shape[-1],
            _lib.stream_handle(h.device)), "vmi_halting_update")

    def accepts(self, out: torch.Tensor, h: torch.Tensor) -> bool:
        return (fusable(out) and out.dtype == h.dtype and out.device == h.device and out.shape == h.shape
                and _rows(out, h))

    def step(self, out, h, active, below_min_depth: bool):
        """The next (h, active)."""
        h_next, still = torch.empty_like(h), torch.empty_like(active)
        self._run(out, h, h_next, active, still, 1 if below_min_depth else 0)
        return h_next, still

    def finish(self, h, active) -> None:
        self._run(None, h, None, active, None, 2)
