"""The training branch's linear layers: torch's products forward, the weight gradients on this package's own kernel.

``linear(x, *weights)`` is ``x @ cat(weights)^T`` in x's dtype with a backward of its own: the input gradient is one
library product, the weight gradient ``mla_weight_grad`` (transformer.py:208-213, :263, :300 under autograd).  Its sums
reach fp32 weights as fp32: autocast's product rounds them to bf16 and casts them back.

Callers take it only where nothing can tell the difference from ``nn.Linear`` (``takes``); everything else (tracing,
transforms, hooked or replaced submodules, other dtypes) keeps torch's own layers.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _nn_module

from . import kernels


def plain_call(*tensors) -> bool:
    """Whether an autograd.Function may stand in for torch's own operators: eager mode, no dispatch mode, functorch
    transform or forward-mode level, and plain GPU tensors."""
    if torch.compiler.is_compiling() or torch._C._len_torch_dispatch_stack() > 0 \
            or torch._C._functorch.peek_interpreter_stack() is not None \
            or torch.autograd.forward_ad._current_level >= 0:
        return False
    return all((type(t) is torch.Tensor or type(t) is nn.Parameter) and t.is_cuda for t in tensors)


def plain_linear(m: nn.Module) -> bool:
    """Whether calling ``m`` is no more than ``x @ m.weight^T``: an nn.Linear without bias, hooks or an override."""
    return (type(m) is nn.Linear and m.bias is None and type(m._parameters.get("weight")) is nn.Parameter
            and "forward" not in m.__dict__
            and not (m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks)
            and not _nn_module._has_any_global_hook())


def takes(m: nn.Module, x: torch.Tensor) -> bool:
    """Whether ``m(x)`` under autograd may run as ``linear``: a plain layer whose weight is trained, in bf16 arithmetic
    that torch's product accepts (autocast, or x in the weight's dtype)."""
    w = m._parameters.get("weight")
    if w is None or not w.requires_grad or not torch.is_grad_enabled() or not plain_linear(m):
        return False
    if torch.is_autocast_enabled("cuda"):
        ok = torch.get_autocast_dtype("cuda") == torch.bfloat16 and w.dtype in (torch.bfloat16, torch.float32)
    else:
        ok = w.dtype == torch.bfloat16 and x.dtype == w.dtype
    return ok and plain_call(x, w)


def cat_weights(weights, dtype):
    """The weights' rows below each other in ``dtype`` (one pass over each, casts included)."""
    if len(weights) == 1:
        return weights[0].detach().to(dtype)
    W = torch.empty(sum(w.size(0) for w in weights), weights[0].size(1), dtype=dtype, device=weights[0].device)
    r = 0
    for w in weights:
        W[r:r + w.size(0)].copy_(w.detach())
        r += w.size(0)
    return W


def weight_grads(dy, x, weights, needed):
    """The gradients (rows of one product ``dy^T x``) of ``weights`` in their own dtypes; None where not ``needed``."""
    if not any(needed):
        return [None] * len(weights)
    f32 = all(w.dtype == torch.float32 for w in weights)
    sy, sx = dy.stride(0), x.stride(0)
    if dy.dtype == torch.bfloat16 and kernels.weight_grad_fits(dy.size(0), dy.size(1), x.size(1), sy, sx):
        dW = kernels.weight_grad(dy, x, f32)
    else:
        dW = torch.matmul(dy.t(), x)
    out, r = [], 0
    for w, need in zip(weights, needed):
        out.append(dW[r:r + w.size(0)].to(w.dtype) if need else None)
        r += w.size(0)
    return out


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, product, *weights):
        W = cat_weights(weights, x.dtype)
        ctx.save_for_backward(x, W)
        ctx.weights = weights
        return product(x, W)

    @staticmethod
    def backward(ctx, dy):
        x, W = ctx.saved_tensors
        weights = ctx.weights
        if torch.is_grad_enabled():  # the backward is itself differentiated: torch's operators on the inputs
            W = torch.cat(weights, 0).to(x.dtype)
            dx = torch.matmul(dy, W)
            dW = torch.matmul(dy.reshape(-1, dy.size(-1)).t(), x.reshape(-1, x.size(-1)))
            return (dx, None) + tuple(g.to(w.dtype) for g, w in zip(dW.split([w.size(0) for w in weights]), weights))
        dx = torch.matmul(dy, W) if ctx.needs_input_grad[0] else None
        grads = weight_grads(dy.reshape(-1, dy.size(-1)), x.reshape(-1, x.size(-1)), weights, ctx.needs_input_grad[2:])
        return (dx, None, *grads)


def linear(x: torch.Tensor, *weights, product=torch.nn.functional.linear) -> torch.Tensor:
    """``product(x, cat(weights))``, by default ``x @ cat(weights)^T``, in x's dtype; see the module."""
    return _Linear.apply(x, product, *weights)
