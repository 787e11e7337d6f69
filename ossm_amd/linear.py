"""Projections over many rows, with their weight gradients on this library's kernel.

``rows_product(a, b)`` is ``a^T b`` for row-major ``a`` [R, M] and ``b`` [R, N]
with R (every batch row and step) much larger than M and N
(``ossm_rows_product``).  ``linear(module, x)`` is ``module(x)`` for an
``nn.Linear`` whose backward takes the weight gradient from it.
"""

from __future__ import annotations

from typing import Optional

import torch
import torch.nn.functional as F
from torch import Tensor, nn

from . import _lib

__all__ = ["rows_product", "linear", "linear_weight", "LinearFn", "is_plain",
           "MIN_ROWS", "BLOCK_ROWS"]

# The least the kernel takes, and where the layers' and the mixer's own backwards, which
# have no operation of torch's to fall back on but transposed products and copies, take
# it: training steps of [rows, 64] at 16 to 400 rows, LinOSS layer 162 us against 196 to
# 292 with those, mixer 519 against 526 to 528.
BLOCK_ROWS = 16
# LinearFn leaves fewer rows to torch: the weight gradient alone then takes 9 us against
# 12 at 200 rows, 60 against 14 at 1000 ([R, 80] x [R, 40] and [R, 256] x [R, 64]).
MIN_ROWS = 512


def _tiles(m: int, n: int) -> int:
    """128 x 64 output tiles of an [m, n] product."""
    return -(-m // 128) * -(-n // 64)


def rows_product(a: Tensor, b: Tensor, pairs: bool = False) -> Tensor:
    """``sum_r a[r, m] b[r, n]`` as [M, N], or with ``pairs`` (M even) as
    [M / 2, N, 2], the rows 2i and 2i + 1 side by side.  float32 on one GPU; any
    row stride, unit column stride (else copied)."""
    if a.dim() != 2 or b.dim() != 2 or a.size(0) != b.size(0):
        raise RuntimeError(f"rows_product: expected [R, M] and [R, N], got {tuple(a.shape)}, {tuple(b.shape)}")
    if a.dtype != torch.float32 or b.dtype != torch.float32 or not a.is_cuda or a.device != b.device:
        raise RuntimeError("rows_product needs float32 tensors on one GPU")
    R, M, N = a.size(0), a.size(1), b.size(1)
    if pairs and M % 2 != 0:
        raise RuntimeError("rows_product: pairs needs an even number of columns in a")
    if R < BLOCK_ROWS or M == 0 or N == 0:
        out = a.t() @ b
        return out.reshape(M // 2, 2, N).transpose(1, 2).contiguous() if pairs else out
    a, b = (t if t.stride(1) == 1 and t.stride(0) >= t.size(1) else t.contiguous() for t in (a, b))
    out = torch.empty((M // 2, N, 2) if pairs else (M, N), dtype=torch.float32, device=a.device)
    strides = (2 * N, 1, 2) if pairs else (2 * N, N, 1)
    if not pairs and _tiles(N, M) < _tiles(M, N):  # the wider side of the tile along N
        a, b, M, N, strides = b, a, N, M, (2, 1, N)
    _lib.run(_lib.load().ossm_rows_product, a, a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0),
             out.data_ptr(), *strides, R, M, N)
    return out


class LinearFn(torch.autograd.Function):
    """``F.linear`` (the library's GEMM) whose weight gradient is ``rows_product``."""

    @staticmethod
    def forward(ctx, x: Tensor, weight: Tensor, bias: Optional[Tensor]) -> Tensor:  # type: ignore[override]
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return F.linear(x, weight, bias)

    @staticmethod
    def backward(ctx, grad: Tensor):  # type: ignore[override]
        x, weight = ctx.saved_tensors
        need_x, need_w, need_b = ctx.needs_input_grad
        g2, x2 = grad.reshape(-1, weight.size(0)), x.reshape(-1, weight.size(1))
        gx = grad @ weight if need_x else None
        gw = None
        if need_w:
            # create_graph: an operation that is differentiable again
            gw = g2.t() @ x2 if torch.is_grad_enabled() else rows_product(g2, x2)
        return gx, gw, (g2.sum(0) if need_b and ctx.has_bias else None)


def is_plain(module: nn.Module) -> bool:
    """Whether calling ``module`` is F.linear on its own weight and nothing else
    (no subclass, no hooks, its own or global, no replaced forward)."""
    glob = nn.modules.module
    return (type(module) is nn.Linear and "forward" not in module.__dict__
            and not (module._forward_hooks or module._forward_pre_hooks or module._backward_hooks
                     or module._backward_pre_hooks or glob._global_forward_hooks
                     or glob._global_forward_pre_hooks or glob._global_backward_hooks
                     or glob._global_backward_pre_hooks))


def linear(module: nn.Module, x: Tensor) -> Tensor:
    """``module(x)``; a plain float32 ``nn.Linear`` on the GPU that trains takes
    its weight gradient from ``rows_product``."""
    if is_plain(module):
        return linear_weight(x, module.weight, module.bias, module)
    return module(x)


def linear_weight(x: Tensor, weight: Tensor, bias: Optional[Tensor] = None,
                  module: Optional[nn.Module] = None) -> Tensor:
    """``F.linear(x, weight, bias)`` (or ``module(x)``), the weight gradient as in ``linear``."""
    if (torch.is_grad_enabled() and weight.requires_grad and type(x) in (Tensor, nn.Parameter)
            and type(weight) in (Tensor, nn.Parameter) and weight.is_cuda and x.device == weight.device
            and x.dtype == weight.dtype == torch.float32 and x.dim() >= 2
            and (bias is None or bias.dtype == torch.float32) and x.numel() >= MIN_ROWS * x.size(-1) > 0
            and weight.size(0) > 0 and not torch.is_autocast_enabled("cuda")
            and not torch.compiler.is_compiling()):
        return LinearFn.apply(x, weight, bias)
    return F.linear(x, weight, bias) if module is None else module(x)
