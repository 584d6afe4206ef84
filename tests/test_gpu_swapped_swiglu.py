"""A SwiGLU block after ``swap_mxfp8`` runs as one graph (``mxfp8_swiglu_pair``): every output against the same block run
layer by layer, over ragged and single rows, types, autocast, frozen weights and views; and who is left to run layer by layer.

Tolerance: both do the same arithmetic on the same 16-bit values, but the graph's sigmoid is the hardware exponential's, so a
share of the 16-bit intermediates (up to 1e-3) rounds the other way and may move an e4m3 code by one step (1/16 of its value at
most): sqrt(1e-3) / 16 = 2e-3 of a product's norm; K slices and batches add 1e-6."""

import pytest
import torch
import torch.nn.functional as F

from conftest import SEED

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _block(dtype, dim=256, hidden=384):
    from kohakuwullm_amd.models.mlp import SwiGLU
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    torch.manual_seed(SEED)
    block = SwiGLU(dim, hidden=hidden).to(DEV).to(dtype)
    swap_mxfp8(block)
    return block


def _step(block, x, dy, autocast):
    leaf = x.detach().requires_grad_(True)
    for p in block.parameters():
        p.grad = None
    with torch.autocast("cuda", dtype=autocast or BF, enabled=autocast is not None):
        y = block(leaf)
    y.backward(dy.to(y.dtype).expand_as(y))
    return [y.detach(), leaf.grad, *(p.grad for p in block.parameters())]


@pytest.mark.parametrize("shape,dtype,autocast,frozen", [
    ((1, 256), BF, None, ()), ((129, 256), HF, None, ()), ((2, 100, 256), BF, None, ()), ((700, 256), F32, BF, ()),
    ((513, 256), F32, HF, ()), ((160, 256), BF, HF, ()), ((200, 256), BF, None, ("w_in",)), ((200, 256), F32, BF, ("w_in", "w_out")),
])
def test_pair_equals_the_layers(oracle, monkeypatch, shape, dtype, autocast, frozen):
    import kohakuwullm_amd.models.mlp as mlp

    block = _block(dtype)
    for name in frozen:
        getattr(block, name).weight.requires_grad_(False)
    g = torch.Generator().manual_seed(SEED)
    x = torch.randn(*shape, generator=g).to(DEV, dtype)
    dy = (torch.randn(*shape, generator=g) * 1e-2).to(DEV)
    calls = []
    pair = mlp.mxfp8_swiglu_pair
    monkeypatch.setattr(mlp, "mxfp8_swiglu_pair", lambda *a: calls.append(pair(*a)) or calls[-1])
    fused = _step(block, x, dy, autocast)
    assert calls and calls[0] is not None
    monkeypatch.setattr(mlp, "mxfp8_swiglu_pair", lambda *a: None)
    layers = _step(block, x, dy, autocast)
    for a, b in zip(fused, layers):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape
            assert oracle.rel_error(a.double().cpu(), b.double().cpu()) < 2e-3


def test_pair_takes_views():
    block = _block(BF)
    wide = torch.randn(96, 520, device=DEV).to(BF)
    assert torch.equal(block(wide[:, 3:259]), block(wide[:, 3:259].contiguous()))
    assert torch.equal(block(wide[:, :256].reshape(2, 48, 256).transpose(0, 1)).transpose(0, 1).reshape(96, 256), block(wide[:, :256]))


def test_who_runs_layer_by_layer():
    from kohakuwullm_amd.kernels.mxfp8.mlp import mxfp8_swiglu_pair

    block = _block(F32)
    x = torch.randn(64, 256, device=DEV)
    pair = lambda x: mxfp8_swiglu_pair(x, block.w_in, block.w_out)  # noqa: E731
    assert pair(x) is None and block(x).dtype == F32  # fp32 without autocast
    assert pair(x.bfloat16()) is not None and pair(x.bfloat16()[:0]) is None
    seen = []
    handle = block.w_out.register_forward_pre_hook(lambda m, args: seen.append(args[0]))
    y = block(x.bfloat16())
    assert len(seen) == 1 and seen[0].shape == (64, 384)
    handle.remove()
    assert pair(x.bfloat16()) is not None and torch.equal(block(x.bfloat16()).isnan(), y.isnan())
    # another activation, a projection of its own kind
    block.act = F.gelu
    assert block(x.bfloat16()).isfinite().all() and not torch.equal(block(x.bfloat16()), pair(x.bfloat16()))


def test_forward_alone_is_the_training_forward():
    """Without gradients only the row-axis operands are made; the result is the training forward's, bit for bit."""
    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear
    from kohakuwullm_amd.models.mlp import MXFP8SwiGLU

    for module in (_block(BF), MXFP8Linear(256, 200).to(DEV), MXFP8SwiGLU(256, hidden=384).to(DEV)):
        for x, autocast in ((torch.randn(77, 256, device=DEV).to(BF), False), (torch.randn(77, 256, device=DEV), True)):
            with torch.autocast("cuda", dtype=BF, enabled=autocast):
                want = module(x.requires_grad_(True)).detach()
                with torch.no_grad():
                    assert torch.equal(module(x), want)
                with torch.inference_mode():
                    assert torch.equal(module(x), want)
