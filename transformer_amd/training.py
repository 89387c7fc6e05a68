"""The training branch's linear layers: torch's products forward, the weight gradients on this package's own kernel.

``linear(x, *weights)`` is ``x @ cat(weights)^T`` in x's dtype with a backward of its own: the input gradient is one
library product, the weight gradient ``mla_weight_grad`` (transformer.py:208-213, :263, :300 under autograd).  Its sums
reach fp32 weights as fp32: autocast's product rounds them to bf16 and casts them back.

``attention`` is everything between the down-projections' output and o_proj's input (transformer.py:208, :228-239,
:306-315), as one Function whose backward writes each part of the down-projections' gradient where their product reads
it.

Callers take them only where nothing can tell the difference from ``nn.Linear`` (``takes``, ``takes_attention``);
everything else (tracing, transforms, hooked or replaced submodules, other dtypes) keeps torch's own layers.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _nn_module

from . import kernels


def plain_call(*tensors) -> bool:
    """Whether an autograd.Function may stand in for torch's own operators on ``tensors`` (see kernels.function_fits)."""
    return kernels.function_fits(tensors)


def plain_linear(m: nn.Module) -> bool:
    """Whether calling ``m`` is no more than ``x @ m.weight^T``: an nn.Linear without bias, hooks or an override."""
    if type(m) is not nn.Linear:
        return False
    d = m.__dict__  # (a decode step asks on every call: attribute lookups on a module take twice as long)
    p = d["_parameters"]
    return (type(p.get("weight")) is nn.Parameter and p.get("bias") is None and "forward" not in d
            and not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"])
            and not _nn_module._has_any_global_hook())


def takes(m: nn.Module, x: torch.Tensor) -> bool:
    """Whether ``m(x)`` under autograd may run as ``linear``: a plain layer whose weight is trained, in bf16 arithmetic
    that torch's product accepts (autocast, or x in the weight's dtype)."""
    w = m._parameters.get("weight")
    return (w is not None and w.requires_grad and torch.is_grad_enabled() and _bf16_arithmetic(m, x)
            and plain_call(x, w))


_AUTOCAST_INPUTS = (torch.bfloat16, torch.float16, torch.float32)  # what autocast casts (float64 it leaves)


def _bf16_arithmetic(m: nn.Module, x: torch.Tensor) -> bool:
    if not plain_linear(m):
        return False
    w = m._parameters["weight"]
    if torch.is_autocast_enabled("cuda"):
        return torch.get_autocast_dtype("cuda") == torch.bfloat16 and x.dtype in _AUTOCAST_INPUTS \
            and w.dtype in (torch.bfloat16, torch.float32)
    return w.dtype == torch.bfloat16 and x.dtype == w.dtype


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
    dW = kernels.weight_grad_or_none(dy, x, f32) if dy.dtype == torch.bfloat16 else None
    if dW is None:
        dW = torch.matmul(dy.t(), x)
    out, r = [], 0
    for w, need in zip(weights, needed):
        out.append(dW[r:r + w.size(0)].to(w.dtype) if need else None)
        r += w.size(0)
    return out


def _by_operators(grad) -> bool:
    """Whether a backward runs through operators that autograd and transforms see: it is itself differentiated, or
    called with a batch of gradients (is_grads_batched) or under a dispatch mode."""
    return torch.is_grad_enabled() or kernels.batched_grad(grad) or kernels._not_plain((grad,))


class _Kept(torch.autograd.Function):
    """The forward's copy of ``weights`` (their rows below each other, cast), whose gradient goes to the weights: an
    operator backward sees the values that the forward saw, whatever has been written to the weights since."""

    @staticmethod
    def forward(ctx, W, *weights):
        ctx.parts = [(w.size(0), w.dtype) for w in weights]
        return W.view_as(W)

    @staticmethod
    def backward(ctx, g):
        rows = g.split([n for n, _ in ctx.parts])
        return (None, *(r.to(dt) for r, (_, dt) in zip(rows, ctx.parts)))


def on_rows(product, x, W):
    """``product(x, W) [rows, N]`` over x's rows as one matrix.  torch's own product of a batch whose rows are not evenly
    spaced (a slice of longer sequences, a transpose) with a weight that needs no gradient is a batched one over the
    expanded transpose of the weight: slow, and bf16 batched products with a transposed right operand have faulted on
    this GPU."""
    return product(x.reshape(-1, x.size(-1)), W)


class _Linear(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, product, *weights):
        W = cat_weights(weights, x.dtype)
        ctx.save_for_backward(x, W)
        ctx.weights = weights
        # (no view, as torch's own output is none: callers may change it in place)
        return torch.ops.aten._unsafe_view.default(on_rows(product, x, W), (*x.shape[:-1], W.size(0)))

    @staticmethod
    def backward(ctx, dy):
        x, W = ctx.saved_tensors
        weights = ctx.weights
        dy2, x2 = dy.reshape(-1, dy.size(-1)), x.reshape(-1, x.size(-1))
        if _by_operators(dy):  # torch's operators on the inputs
            W = _Kept.apply(W, *weights)
            dx = torch.matmul(dy2, W).view(x.shape)
            dW = torch.matmul(dy2.t(), x2)
            return (dx, None) + tuple(g.to(w.dtype) for g, w in zip(dW.split([w.size(0) for w in weights]), weights))
        dx = torch.matmul(dy2, W).view(x.shape) if ctx.needs_input_grad[0] else None
        return (dx, None, *weight_grads(dy2, x2, weights, ctx.needs_input_grad[2:]))


def linear(x: torch.Tensor, *weights, product=torch.nn.functional.linear) -> torch.Tensor:
    """``product(x, cat(weights))``, by default ``x @ cat(weights)^T``, in x's dtype; see the module."""
    return _Linear.apply(x, product, *weights)


class _Attention(torch.autograd.Function):
    """d [B, T, q_lora + (H + hr) 64 + d_latent], the down-projections' output -> o [B, T, H d_v].

    The up-projections of the latent run as one product over [W_UK; W_UV], K and V the column views of its result.  In
    the backward, dq_rope, dk_rope and the two products' results go straight to their columns of d's gradient, and dK
    and dV to theirs of one buffer: one product gives the latent's gradient (dK W_UK + dV W_UV in one fp32 sum) and one
    the weights'.  As separate nodes, autograd filled, copied, added and concatenated full-size tensors around them:
    107 of 1495 us of a training pass of one block (default dims, B = 6, T = 2048)."""

    @staticmethod
    def forward(ctx, d, Wq, Wk, Wv, cos, sin, layout, scale):
        H, dn, dv, hr, ql, dl = layout
        with kernels.below_autograd():
            B, T, n = d.shape
            d2 = d.reshape(B * T, n)
            Wqb, Wkv = cat_weights((Wq,), d.dtype), cat_weights((Wk, Wv), d.dtype)
            qk = d2[:, ql:n - dl].view(B, T, H + hr, 64)
            q = torch.mm(d2[:, :ql], Wqb.t()).view(B, T, H, dn)
            kv = torch.mm(d2[:, n - dl:], Wkv.t())
            k_nope, v = _kv_views(kv, B, T, H, dn, dv)
            k_rope = kernels.eager.rope(qk[:, :, H:], cos, sin, 0, False)
            o, lse, q_rot = kernels.eager.prefill_fwd_rope(q, qk[:, :, :H], k_nope, k_rope, v, cos, sin, scale, True, 0,
                                                           0, True)
        ctx.save_for_backward(d, Wqb, Wkv, q, q_rot, kv, k_rope, o, lse, cos, sin)
        ctx.weights, ctx.layout, ctx.scale = (Wq, Wk, Wv), layout, scale
        return o.view(B, T, H * dv)

    @staticmethod
    def backward(ctx, do):
        d, Wqb, Wkv, q, q_rot, kv, k_rope, o, lse, cos, sin = ctx.saved_tensors
        H, dn, dv, hr, ql, dl = ctx.layout
        B, T, n = d.shape
        if _by_operators(do):
            with torch.enable_grad():
                Wq, Wkv = _Kept.apply(Wqb, ctx.weights[0]), _Kept.apply(Wkv, *ctx.weights[1:])
                out = _attention_by_operators(d, Wq, Wkv, cos, sin, ctx.layout, ctx.scale)
            # (with respect to the copies: k_up and v_up may be one tied weight)
            got = iter(torch.autograd.grad(out, [t for t in (d, Wq, Wkv) if t.requires_grad], do,
                                           create_graph=torch.is_grad_enabled()))
            gd, gq, gkv = (next(got) if t.requires_grad else None for t in (d, Wq, Wkv))
            gk, gv = gkv.split([H * dn, H * dv]) if gkv is not None else (None, None)
            grads = [g.to(w.dtype) if need else None
                     for g, w, need in zip((gq, gk, gv), ctx.weights, ctx.needs_input_grad[1:4])]
            return (gd, *grads) + (None,) * 4
        d2 = d.reshape(B * T, n)
        dd = torch.empty(B * T, n, dtype=d.dtype, device=d.device)
        dqk = dd[:, ql:n - dl].view(B, T, H + hr, 64)
        dq = torch.empty(B, T, H, dn, dtype=d.dtype, device=d.device)
        dkv = torch.empty_like(kv)
        dk_nope, dvv = _kv_views(dkv, B, T, H, dn, dv)
        k_nope, v = _kv_views(kv, B, T, H, dn, dv)
        kernels._prefill_bwd_impl(do.reshape(B, T, H, dv), q, q_rot, k_nope, k_rope, v, o, lse, ctx.scale, True, 0, cos,
                                  sin, 0, out=(dq, dqk[:, :, :H], dk_nope, dqk[:, :, H:], dvv))
        kernels.eager.rope_(dqk[:, :, H:], cos, sin, 0, True)
        dq2 = dq.view(B * T, H * dn)
        if ctx.needs_input_grad[0]:
            torch.mm(dq2, Wqb, out=dd[:, :ql])
            torch.mm(dkv, Wkv, out=dd[:, n - dl:])
        (Wq, Wk, Wv), (_, nq, nk, nv) = ctx.weights, ctx.needs_input_grad[:4]
        (gq,) = weight_grads(dq2, d2[:, :ql], (Wq,), (nq,))
        gk, gv = weight_grads(dkv, d2[:, n - dl:], (Wk, Wv), (nk, nv))
        return dd.view(B, T, n) if ctx.needs_input_grad[0] else None, gq, gk, gv, None, None, None, None


def _kv_views(kv, B, T, H, dn, dv):
    """K_nope [B, T, H, dn] and V [B, T, H, dv] in the columns of ``kv [B T, H (dn + dv)]``."""
    return kv[:, :H * dn].view(B, T, H, dn), kv[:, H * dn:].view(B, T, H, dv)


def _attention_by_operators(d, Wq, Wkv, cos, sin, layout, scale):
    H, dn, dv, hr, ql, dl = layout
    B, T, n = d.shape
    q_low, qk, kv = d.split([ql, (H + hr) * 64, dl], -1)
    lin = torch.nn.functional.linear
    qk = qk.view(B, T, H + hr, 64)
    Wk, Wv = Wkv.split([H * dn, H * dv])
    q, k, v = (lin(t, w).view(B, T, H, -1) for t, w in ((q_low, Wq), (kv, Wk), (kv, Wv)))
    k_rope = kernels.eager.rope(qk[:, :, H:], cos, sin, 0, False)
    o, _, _ = kernels.eager.prefill_fwd_rope(q, qk[:, :, :H], k, k_rope, v, cos, sin, scale, True, 0, 0, True)
    return o.reshape(B, T, H * v.size(-1))


def takes_attention(mla, d: torch.Tensor) -> bool:
    """Whether ``attention`` may run the no-cache branch on the down-projections' bf16 output ``d``: its gradient or a
    weight's is needed, the three layers are plain in bf16 arithmetic, and every part of ``d`` is whole 16-byte runs."""
    mods = [mla._modules[n] for n in ("q_up", "k_up", "v_up")]
    # (plain layers first: nothing else is known to have a weight)
    if not (torch.is_grad_enabled() and d.dtype == torch.bfloat16 and d.numel() > 0
            and all(_bf16_arithmetic(m, d) for m in mods)
            and mla.d_latent % 8 == 0 and mods[0].in_features % 8 == 0
            and mla.content_dim in kernels.SUPPORTED_NOPE and mla.v_head_dim in kernels.SUPPORTED_V):
        return False
    ws = [m.weight for m in mods]
    return (d.requires_grad or any(w.requires_grad for w in ws)) and plain_call(d, *ws)


def attention(mla, d: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """o_proj's input from the down-projections' output, causal over its own positions; see ``_Attention``."""
    q, k, v = (mla._modules[n].weight for n in ("q_up", "k_up", "v_up"))
    layout = (mla.n_heads, mla.content_dim, mla.v_head_dim, mla.n_k_rope_heads, q.size(1), mla.d_latent)
    return _Attention.apply(d, q, k, v, cos, sin, layout, mla.scale)
