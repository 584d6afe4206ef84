"""Sigmoid top-k routing on the HIP kernels: scores, selection, gate weights and histogram in one pass, with its backward.

Counterpart of ``TopKRouter.route`` (``src/kohakuwullm/models/components/moe.py:97-199``) for a router without groups and
auxiliary losses; :class:`kohakuwullm_amd.models.moe.TopKRouter` uses it where :func:`can_route` allows and its PyTorch
composition elsewhere.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch.autograd import forward_ad

from kohakuwullm_amd import _lib, host
from kohakuwullm_amd.kernels.mxfp8.quantize import aligned_rows

MAX_EXPERTS, MAX_TOP_K = 256, 16
MAX_TOKENS, MAX_WIDTH = 65535 * 256, (1 << 24) - 1  # the backward's grid has 65535 chunks of 256 tokens at most


def operands_fit(x: torch.Tensor, weight: torch.Tensor, top_k: int, bias: torch.Tensor | None = None) -> bool:
    """Whether shapes, types and layouts are what the kernels assume; the library sees pointers and cannot check a width."""
    if x.dim() != 2 or weight.dim() != 2:
        return False
    e, d = weight.shape
    if bias is not None and not (bias.shape == (e,) and bias.dtype in _lib.MX_DTYPE and bias.is_contiguous() and bias.device == x.device):
        return False
    return (0 < x.shape[0] <= MAX_TOKENS and x.shape[1] == d <= MAX_WIDTH and x.dtype in _lib.MX_DTYPE and weight.dtype in (x.dtype, torch.float32)
            and d % 8 == 0 and e <= MAX_EXPERTS and 0 < top_k <= min(MAX_TOP_K, e) and weight.is_contiguous()
            and weight.device == x.device and weight.data_ptr() % 16 == 0)


def plain_call(*tensors: torch.Tensor) -> bool:
    """Whether an autograd function may stand for the operators it replaces: nobody traces them (torch.compile, torch.jit, dispatch
    modes), transforms them (vmap, torch.func, forward mode) or dispatches them itself (tensor subclasses).  A gradient mapped by
    ``is_grads_batched`` shows by its missing storage alone: its backward runs on a thread that knows of no transform."""
    return not (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._are_functorch_transforms_active()
                or forward_ad._current_level >= 0 or torch._C._len_torch_dispatch_stack()
                or any(type(t) not in (torch.Tensor, torch.nn.Parameter) or not torch._C._has_storage(t) for t in tensors))


def can_route(x: torch.Tensor, weight: torch.Tensor, top_k: int, bias: torch.Tensor | None = None) -> bool:
    """Whether the kernels take this call; autocast changes the arithmetic and is not covered."""
    return (plain_call(x, weight) and x.is_cuda and operands_fit(x, weight, top_k, bias)
            and not torch.is_autocast_enabled("cuda"))


def composed_gradients(grad, x, weight, idx, norm: bool, factor: float):
    """``(dx, dweight)`` of the gate weights by PyTorch operators, for backwards that are themselves differentiated or mapped."""
    scores = F.linear(x.float(), weight.float()).sigmoid()
    picked, g = scores.gather(1, idx), grad.float() * factor
    if norm:
        total = picked.sum(-1, keepdim=True)
        unit = total.clamp_min(1e-9)
        along = (g * picked).sum(-1, keepdim=True) / unit
        g = (g - torch.where(total < 1e-9, torch.zeros_like(along), along)) / unit
    dlogit = torch.zeros_like(scores).scatter(1, idx, g * picked * (1.0 - picked))
    return (dlogit @ weight.float()).to(x.dtype), (dlogit.transpose(0, 1) @ x.float()).to(weight.dtype)


class _RouteTopK(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, top_k, norm, factor, through=False):
        (t, d), e, dev = x.shape, weight.shape[0], x.device
        need = ctx.needs_input_grad[0] or ctx.needs_input_grad[1]
        made = host.route_forward(x, weight, bias, top_k, norm, factor, need)
        if made is None:
            idx = torch.empty(t, top_k, device=dev, dtype=torch.int64)
            gate = torch.empty(t, top_k, device=dev, dtype=x.dtype)
            scores = torch.empty(t, top_k, device=dev, dtype=torch.float32) if need else None
            counts = torch.empty(e, device=dev, dtype=torch.int32)
            _lib.invoke(
                "mx_router_topk", 2.0 * t * d * e, x, x.data_ptr(), _lib.MX_DTYPE[x.dtype], x.stride(0), weight.data_ptr(),
                _lib.MX_DTYPE[weight.dtype], 0 if bias is None else bias.data_ptr(), 0 if bias is None else _lib.MX_DTYPE[bias.dtype],
                t, d, e, top_k, int(norm), float(factor), idx.data_ptr(), gate.data_ptr(), 0 if scores is None else scores.data_ptr(),
                counts.data_ptr(),
            )
        else:
            idx, gate, scores, counts = made
        if need:
            ctx.save_for_backward(x, weight, idx, scores)
            ctx.norm, ctx.factor = norm, factor
        ctx.mark_non_differentiable(idx, counts)
        ctx.set_materialize_grads(False)
        return (idx, gate, counts, x) if through else (idx, gate, counts)

    @staticmethod
    def backward(ctx, _idx, grad, _counts, onto=None):
        rest = (None,) * 5
        if not ctx.needs_input_grad[0]:
            onto = None
        if grad is None:
            return onto, None, *rest
        x, weight, idx, scores = ctx.saved_tensors
        if torch.is_grad_enabled() or not plain_call(grad, *(() if onto is None else (onto,))):
            # create_graph; a vmap over upstream gradients
            dx, dw = composed_gradients(grad, x, weight, idx, ctx.norm, ctx.factor)
            dx = dx if onto is None else dx + onto
            return dx if ctx.needs_input_grad[0] else None, dw if ctx.needs_input_grad[1] else None, *rest
        made = host.route_backward(grad, x, weight, idx, scores, ctx.norm, ctx.factor, *ctx.needs_input_grad[:2], onto)
        if made is not None:
            return *made, *rest
        # as they were saved, unless a saved-tensor hook laid them out anew
        x, weight, idx, scores = aligned_rows(x), aligned_rows(weight.contiguous()), idx.contiguous(), scores.contiguous()
        (t, d), e, lib = x.shape, weight.shape[0], _lib.load()
        grad = grad.contiguous()
        dx = torch.empty(t, d, device=x.device, dtype=x.dtype) if ctx.needs_input_grad[0] else None
        dw = torch.empty_like(weight) if ctx.needs_input_grad[1] else None
        words = lib.mx_router_backward_workspace(t, d, e) if dw is not None else 0
        scratch = torch.empty(words, device=x.device, dtype=torch.float32)
        onto = None if onto is None else aligned_rows(onto)
        below = () if onto is None else (onto.data_ptr(), onto.stride(0))
        _lib.invoke(
            "mx_router_topk_backward_onto" if below else "mx_router_topk_backward", 4.0 * t * d * e, x, *below, grad.data_ptr(), _lib.MX_DTYPE[grad.dtype], idx.data_ptr(),
            scores.data_ptr(), x.data_ptr(), _lib.MX_DTYPE[x.dtype], x.stride(0), weight.data_ptr(), _lib.MX_DTYPE[weight.dtype],
            t, d, e, idx.shape[1], int(ctx.norm), float(ctx.factor), 0 if dx is None else dx.data_ptr(), d,
            0 if dw is None else dw.data_ptr(), scratch.data_ptr() if words else 0, words,
        )
        return dx, dw, *rest


def route_topk(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None, top_k: int, norm: bool, factor: float):
    """``(idx (T, k) int64, gate (T, k) in x's type, counts (E,) int32)`` of sigmoid scores ``x @ weight.T``.

    The ``top_k`` experts with the largest ``score + bias``, best first (ties to the lower expert); ``gate`` is ``factor``
    times their scores, normalized over the token's picks when ``norm``.  Differentiable in ``x`` and ``weight`` through
    ``gate``.  See :func:`can_route` for what it takes; other operands are refused here.
    """
    if not operands_fit(x, weight, top_k, bias):
        raise ValueError(f"route_topk: x {tuple(x.shape)} {x.dtype}, weight {tuple(weight.shape)} {weight.dtype}, top_k {top_k}, "
                         f"bias {None if bias is None else (tuple(bias.shape), bias.dtype, bias.device)}")
    return route_fitting(x, weight, bias, top_k, norm, factor)


def route_fitting(x, weight, bias, top_k: int, norm: bool, factor: float, through: bool = False):
    """:func:`route_topk` of operands that :func:`can_route` has just looked at (a second look takes 2.6 us).

    ``through``: ``x`` is returned behind the results, for whoever computes on it next.  Its gradient then comes through the
    router's node, whose kernel adds its own to it: one rounding, and no launch to add the two."""
    # a copied input is copied in front of the graph's node, which then keeps the tensor it differentiates
    x = aligned_rows(x)
    if host.unrecorded(x, weight):
        made = host.route_forward(x, weight, bias, top_k, norm, factor, False)
        if made is not None:
            return (made[0], made[1], made[3], x) if through else (made[0], made[1], made[3])
    return _RouteTopK.apply(x, weight, bias, top_k, norm, factor, through)
