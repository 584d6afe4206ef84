"""Dense SwiGLU feed-forward in MXFP8 with the activation fused into the quantizers.

The reference's dense ``GLUMLP`` runs ``w_out(silu(gate) * value)`` as two ``MXFP8Linear``
calls around an eager 16-bit activation (``src/kohakuwullm/models/components/mlp.py:68-73``)
and names the fused cast ``swiglu_mx`` (``kernels/mxfp8/fused_act.py:69-101``) as the
producer epilogue it wants.  This function is that fusion for the whole layer:

forward   X --dual quantize--> GU = Xq . Wq_in^T --SwiGLU + dual quantize--> Y = Hq . Wq_out^T
backward  dY --dual quantize--> dH = dYq . Wq_out_d^T --SwiGLU' + dual quantize--> dX = dPq . Wq_in_d^T
          dW_out = dY^T . H^T-blocks,  dW_in = dP^T . X^T-blocks   (contraction over tokens)

``h`` and ``dpre`` never exist in 16 bits: the SwiGLU kernels read the GEMM output once and
emit the row-blocked operand for the next GEMM and the token-blocked operand for WGRAD.
"""

from __future__ import annotations

import torch

from kohakuwullm_amd import _lib, host
from kohakuwullm_amd.kernels.mxfp8.linear import TENSORS, compute_dtype, gradient_dtype, pad_tokens, unobserved
from kohakuwullm_amd.kernels.mxfp8.quantize import (
    BLOCK_SCALE,
    PANEL,
    TILE_ROWS,
    activation_matrix,
    aligned_rows,
    mxfp8_matmul_pq,
    products_by_dtype,
    quantize_mx_dual,
    quantize_tokens,
    stage_major_ok,
    token_axis_buffers,
    token_extent,
)

_FP8 = torch.float8_e4m3fn

# The two projection outputs that only the SwiGLU quantizers read (`gu`, `dh`) are allocated with 128 spare
# elements per row.  Their natural pitches (16 KiB and 8 KiB at the benchmark shape) put the 128 rows a quantizer
# tile reads at once on a few memory channels; 256 bytes more spread them.  Measured in the step at 16384 x 1536 x
# 4096: SwiGLU 75.6 -> 73.1 us, SwiGLU' 135.0 -> 129.4 us, the GEMM that writes `gu` 183.7 -> 186.0 us (64 or 256
# elements: no gain).
_PITCH_PAD = 128


def swiglu_mx_dual(gu: torch.Tensor, stage_major_t: bool = False):
    """``h = silu(gu[:, :H]) * gu[:, H:]`` as ``(q, s, qT, sT)``: blocks along H and along tokens.

    ``stage_major_t``: ``qT`` as ``(tokens // 128, H, 128)`` (see :func:`quantize_mx_dual`).
    """
    m, two_h = gu.shape
    h = two_h // 2
    if two_h % 2 or h % BLOCK_SCALE or m % BLOCK_SCALE:
        raise ValueError(f"gu {tuple(gu.shape)}: tokens and hidden must be multiples of {BLOCK_SCALE}")
    if stage_major_t and not stage_major_ok(m):
        raise ValueError(f"stage_major_t needs the token count {m} to be a positive multiple of {PANEL}")
    _lib.require_gpu(gu, "gu")
    q = torch.empty(m, h, device=gu.device, dtype=_FP8)
    s = torch.empty(m, h // BLOCK_SCALE, device=gu.device, dtype=torch.uint8)
    qt = torch.empty((m // PANEL, h, PANEL) if stage_major_t else (h, m), device=gu.device, dtype=_FP8)
    st = torch.empty(h, m // BLOCK_SCALE, device=gu.device, dtype=torch.uint8)
    _lib.invoke(
        "mx_swiglu_quantize_dual", m * h * (2 * gu.element_size() + 2 * (1 + 1 / BLOCK_SCALE)), gu,
        gu.data_ptr(), _lib.MX_DTYPE[gu.dtype], m, h, gu.stride(0), q.data_ptr(), h, s.data_ptr(), h // BLOCK_SCALE,
        qt.data_ptr(), PANEL if stage_major_t else m, st.data_ptr(), m // BLOCK_SCALE,
    )
    return q, s, qt, st


def swiglu_bwd_mx_dual(dh: torch.Tensor, gu: torch.Tensor, stage_major: bool = False):
    """SwiGLU backward emitted straight in MXFP8: ``dpre = [dgate | dup]`` as ``(q, s, qT, sT)``.

    ``stage_major``: ``q`` as ``(2H // 128, tokens, 128)`` and ``qT`` as ``(MT // 128, 2H, 128)`` with ``MT =
    token_extent(tokens)`` (H a multiple of 128, any token count; see :func:`quantize_tokens`).
    """
    m, two_h = gu.shape
    h = two_h // 2
    if dh.shape != (m, h) or h % BLOCK_SCALE or (m % BLOCK_SCALE and not stage_major):
        raise ValueError(f"dh {tuple(dh.shape)} does not match gu {tuple(gu.shape)}")
    if stage_major and not stage_major_ok(h):
        raise ValueError(f"stage_major needs H={h} to be a positive multiple of {PANEL}")
    _lib.require_gpu(gu, "gu")
    if stage_major:
        return swiglu_bwd_tokens(dh, gu)
    q = torch.empty(m, two_h, device=gu.device, dtype=_FP8)
    s = torch.empty(m, two_h // BLOCK_SCALE, device=gu.device, dtype=torch.uint8)
    qt = torch.empty(two_h, m, device=gu.device, dtype=_FP8)
    st = torch.empty(two_h, m // BLOCK_SCALE, device=gu.device, dtype=torch.uint8)
    _lib.invoke(
        "mx_swiglu_bwd_quantize_dual", m * h * (3 * gu.element_size() + 4 * (1 + 1 / BLOCK_SCALE)), gu,
        dh.data_ptr(), dh.stride(0), gu.data_ptr(), gu.stride(0), _lib.MX_DTYPE[gu.dtype], m, h,
        q.data_ptr(), two_h, s.data_ptr(), two_h // BLOCK_SCALE, qt.data_ptr(), m, st.data_ptr(), m // BLOCK_SCALE,
    )
    return q, s, qt, st


_WHOLE_RANGE: dict = {}


def _whole_range(device, rows: int) -> torch.Tensor:
    """``[0, rows]`` as the offset table of a single "expert" that owns every row (cached: built once)."""
    key = (device, rows)
    if key not in _WHOLE_RANGE:
        _WHOLE_RANGE[key] = torch.tensor([0, rows], dtype=torch.int32, device=device)
    return _WHOLE_RANGE[key]


def fused_swiglu_projection(xq, xs, wq, ws, out_dtype):
    """``gu = x . w_in^T`` with SwiGLU and both casts of ``h`` in the GEMM's epilogue.

    Returns ``gu (M, 2H)`` in ``out_dtype`` (the rounded accumulators, saved for the backward),
    ``h`` quantized along H ``(hq, hs)`` and along the tokens ``(htq, hts)``.  ``h`` is computed
    from the rounded ``gu``, exactly as :func:`swiglu_mx_dual` does on the stored tensor.
    Needs ``M % 128 == 0`` (token-axis tiles) and a 128-multiple contraction.
    """
    from kohakuwullm_amd.kernels.mxfp8.moe import launch_gemm1

    m, k = xq.shape
    hidden = wq.shape[0] // 2
    dev = xq.device
    gu = torch.empty(m, 2 * hidden, device=dev, dtype=out_dtype)
    hq = torch.empty(m, hidden, device=dev, dtype=_FP8)
    hs = torch.empty(m, hidden // BLOCK_SCALE, device=dev, dtype=torch.uint8)
    htq = torch.empty(hidden, m, device=dev, dtype=_FP8)
    hts = torch.empty(hidden, m // BLOCK_SCALE, device=dev, dtype=torch.uint8)
    launch_gemm1(xq, xs, None, wq.unsqueeze(0), ws.unsqueeze(0), hq, hs, gu, _whole_range(dev, m), hidden, k, out_dtype,
                 htq, hts)
    return gu, hq, hs, htq, hts


def swiglu_tokens(gu: torch.Tensor, rounded: bool = False, token_axis: bool = True):
    """``h = silu(gu[:, :H]) * gu[:, H:]`` as ``(q, s, qT, sT)`` for any token count (see :func:`quantize_tokens`).

    ``rounded``: ``silu`` and the product each rounded to the type of ``gu``, the arithmetic of the unfused activation.
    Without ``token_axis`` ``qT`` and ``sT`` are not made and come back as ``None``.
    """
    made = host.swiglu_tokens(gu, rounded, token_axis)
    if made is not None:
        return made
    m, h, dev = gu.shape[0], gu.shape[1] // 2, gu.device
    q = torch.empty(m, h, device=dev, dtype=_FP8)
    s = torch.empty(m, h // BLOCK_SCALE, device=dev, dtype=torch.uint8)
    qt, st, out_t = token_axis_buffers(m, h, dev, token_axis)
    _lib.invoke(
        "mx_swiglu_quantize_tokens", m * h * (2 * gu.element_size() + (1 if qt is None else 2) * (1 + 1 / BLOCK_SCALE)), gu,
        gu.data_ptr(), _lib.MX_DTYPE[gu.dtype], int(rounded), m, h, gu.stride(0), token_extent(m), q.data_ptr(), h,
        s.data_ptr(), h // BLOCK_SCALE, *out_t,
    )
    return q, s, qt, st


def swiglu_bwd_tokens(dh: torch.Tensor, gu: torch.Tensor, rounded: bool = False):
    """``dpre = [dgate | dup]`` as ``(q, s, qT, sT)``, both code matrices stage-major, for any token count (``H % 128 == 0``)."""
    made = host.swiglu_bwd_tokens(dh, gu, rounded)
    if made is not None:
        return made
    gu = aligned_rows(gu)  # as the product wrote it, unless a saved-tensor hook laid it out anew
    m, two_h = gu.shape
    h, dev, mt = two_h // 2, gu.device, token_extent(m)
    q = torch.empty(two_h // PANEL, m, PANEL, device=dev, dtype=_FP8)
    s = torch.empty(m, two_h // BLOCK_SCALE, device=dev, dtype=torch.uint8)
    qt = torch.empty(mt // PANEL, two_h, PANEL, device=dev, dtype=_FP8)
    st = torch.empty(two_h, mt // BLOCK_SCALE, device=dev, dtype=torch.uint8)
    _lib.invoke(
        "mx_swiglu_bwd_quantize_tokens", m * h * (3 * gu.element_size() + 4 * (1 + 1 / BLOCK_SCALE)), gu,
        dh.data_ptr(), dh.stride(0), gu.data_ptr(), gu.stride(0), _lib.MX_DTYPE[gu.dtype], int(rounded), m, h, mt,
        q.data_ptr(), PANEL, s.data_ptr(), two_h // BLOCK_SCALE, qt.data_ptr(), st.data_ptr(), mt // BLOCK_SCALE,
    )
    return q, s, qt, st


def _forward_products(x, compute, in_f, out_f, rounded, wgrad_in, wgrad_out, stage_major):
    """``(y, xtq, xts, gu, htq, hts)`` of the forward, ``y`` with the rows of whole blocks where the operands are row-major."""
    x2d = activation_matrix(x, compute)
    if stage_major:
        xq, xs, xtq, xts = quantize_tokens(x2d, compute, token_axis=wgrad_in)
    else:
        xq, xs, xtq, xts = quantize_mx_dual(pad_tokens(x2d.to(compute)))
    # GEMM, then one bandwidth-bound pass for SwiGLU and both casts: measured faster at the
    # benchmark shape (220 + 89 us) than the same work in the GEMM's epilogue
    # (fused_swiglu_projection: 329 us), whose vector ALU work cannot overlap the MFMAs.
    gu = mxfp8_matmul_pq(xq, xs, *in_f, compute, out_pad=_PITCH_PAD)
    hq, hs, htq, hts = swiglu_tokens(gu, rounded, wgrad_out) if stage_major else swiglu_mx_dual(gu)
    return mxfp8_matmul_pq(hq, hs, *out_f, compute), xtq, xts, gu, htq, hts


class _MXFP8SwiGLUMLP(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w_in, w_out, in_f, in_d, out_f, out_d, rounded, differentiable):
        compute = compute_dtype(x)
        shape = x.shape
        tokens = x.numel() // shape[-1] if shape[-1] else 0
        # The token-axis operands (and dpre below) are written stage-major: each K stage of a tile of the three backward
        # products, which contract over thousands of tokens, is then one contiguous run.  A hidden width that is not
        # whole panels keeps the row-major kernels, which take whole 32-token blocks: zero rows change no gradient.
        sm = stage_major_ok(w_out.shape[1]) and tokens > 0
        wgrad_in, wgrad_out = (need and differentiable for need in ctx.needs_input_grad[1:3])
        made = host.swiglu_mlp_forward(x, compute, in_f, out_f, rounded, wgrad_in, wgrad_out, _PITCH_PAD) if sm else None
        if made is None:
            y, *kept = _forward_products(x, compute, in_f, out_f, rounded, wgrad_in, wgrad_out, sm)
            y = y[:tokens].reshape(*shape[:-1], y.shape[-1])
        else:
            y, *kept = made
        if differentiable and any(ctx.needs_input_grad):
            ctx.save_for_backward(*kept, *in_d, *out_d)
            ctx.compute = compute
            ctx.x_dtype = x.dtype
            ctx.dw_dtypes = gradient_dtype(w_in, compute), gradient_dtype(w_out, compute)
            ctx.stage_major, ctx.rounded = sm, rounded
        return y

    @staticmethod
    def backward(ctx, dout):
        xtq, xts, gu, htq, hts, win_dq, win_ds, wout_dq, wout_ds = ctx.saved_tensors
        shape = dout.shape
        d2d = activation_matrix(dout, ctx.compute)
        tokens = d2d.shape[0]
        if ctx.stage_major:
            dq, ds, dtq, dts = quantize_tokens(d2d, ctx.compute, token_axis=ctx.needs_input_grad[2])
        else:
            dq, ds, dtq, dts = quantize_mx_dual(pad_tokens(d2d.to(ctx.compute)))
        dh = mxfp8_matmul_pq(dq, ds, wout_dq, wout_ds, ctx.compute, out_pad=_PITCH_PAD)
        pq, ps, ptq, pts = swiglu_bwd_tokens(dh, gu, True) if ctx.rounded else swiglu_bwd_mx_dual(dh, gu, stage_major=ctx.stage_major)
        # The last three products are independent and none fills the GPU alone (dW has few
        # tiles with a long K): those of one output type go down together and share the GPU by work.
        wanted = [((pq, ps, win_dq, win_ds), ctx.x_dtype), ((ptq, pts, xtq, xts), ctx.dw_dtypes[0]),
                  ((dtq, dts, htq, hts), ctx.dw_dtypes[1])]
        dx, dw_in, dw_out = products_by_dtype(wanted, ctx.needs_input_grad)
        if dx is not None:
            dx = dx[:tokens].reshape(*shape[:-1], dx.shape[-1])
        return dx, dw_in, dw_out, None, None, None, None, None, None


def _evaluated(x, w_in, w_out, in_f, out_f, rounded) -> torch.Tensor | None:
    """The block's output where no gradient is recorded, without an autograd function around it (``None``: not such a call)."""
    if not stage_major_ok(out_f[0].shape[1]) or not host.unrecorded(x, w_in, w_out):
        return None
    made = host.swiglu_mlp_forward(x, compute_dtype(x), in_f, out_f, rounded, False, False, _PITCH_PAD)
    return None if made is None else made[0]


def mxfp8_swiglu_mlp(x, w_in, w_out, packed) -> torch.Tensor:
    """``(silu(x W_g^T) * (x W_u^T)) W_out^T`` with ``w_in = [W_g; W_u]`` ``(2H, dim)``, ``w_out`` ``(dim, H)``.

    ``packed`` is ``(in_fwd, in_dgrad, out_fwd, out_dgrad)``, each a ``(codes, scales)`` pair:
    the weights blocked along their contraction axis for FPROP and along the other axis for
    DGRAD.  ``w_in``/``w_out`` are passed so autograd routes ``dW`` to the master parameters.
    ``dim`` and ``H`` must be multiples of 32; any token count is taken.
    """
    if w_in.shape[0] != 2 * w_out.shape[1] or w_in.shape[1] != x.shape[-1] or w_out.shape[0] != x.shape[-1]:
        raise ValueError(f"shape mismatch: x {tuple(x.shape)}, w_in {tuple(w_in.shape)}, w_out {tuple(w_out.shape)}")
    y = _evaluated(x, w_in, w_out, packed[0], packed[2], False)
    return _MXFP8SwiGLUMLP.apply(x, w_in, w_out, *packed, False, torch.is_grad_enabled()) if y is None else y


def mxfp8_swiglu_pair(x, w_in, w_out) -> torch.Tensor | None:
    """``w_out(silu(gate) * value)`` of two :class:`MXFP8Linear` around the 16-bit activation, as one graph.

    The activation's two operators and their gradients ran as six library passes over ``(tokens, H)`` or ``(tokens, 2H)``
    matrices, between quantizers that read each result back: 174 us of a 600 us step over 5003 tokens x 1536 x 4096.  Here
    the SwiGLU quantizers do them on the way, with every intermediate rounded as those operators round it.  ``None`` for
    what this graph does not stand for: a layer someone watches (hooks), padded widths, a type other than bf16 / fp16, more
    tokens than its quantizers cover.
    """
    if not (unobserved(w_in) and unobserved(w_out)) or not x.is_cuda or not x.numel() or type(x) not in TENSORS:
        return None
    if x.numel() // x.shape[-1] > TILE_ROWS:
        return None
    compute = compute_dtype(x)
    if compute not in (torch.bfloat16, torch.float16) or x.dtype not in _lib.MX_DTYPE or x.shape[-1] != w_in.in_features:
        return None
    if w_in.out_features != 2 * w_out.in_features or w_out.out_features % PANEL:
        return None
    for lin in (w_in, w_out):
        if lin._cache is None:
            lin.refresh_quantized_weight()
    (in_f, in_d), (out_f, out_d) = ((lin._cache[:2], lin._cache[2:]) for lin in (w_in, w_out))
    y = _evaluated(x, w_in.weight, w_out.weight, in_f, out_f, True)
    if y is not None:
        return y
    return _MXFP8SwiGLUMLP.apply(x, w_in.weight, w_out.weight, in_f, in_d, out_f, out_d, True,
                                 torch.is_grad_enabled())
