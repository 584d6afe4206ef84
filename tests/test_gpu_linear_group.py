"""Projections of one input as one graph (``mxfp8_linear_group``): the quantizer of matrices side by side and the copy that
joins the weights byte for byte, the graph against the same layers one by one, and the calls that stay layer by layer.

Tolerances against the layers: the forward and dW are the same sums of the same codes, K slices apart (one rounding of the
result that goes the other way now and then: 1e-3 in 16 bits, 1e-5 in fp32); a 16-bit dx is rounded once, the layers' shares
(together as large as dx) once each and their two sums once each: four independent roundings of the size of dx or less between
the two, each of at most half an ulp, uniform: 2^-7 / sqrt(12) of the value at most, 2 * 2.3e-3 = 4.6e-3 for the four."""

import pytest
import torch

from conftest import SEED

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _randn(*shape, scale=1.0):
    g = torch.Generator().manual_seed(SEED + shape[0])
    return (torch.randn(*shape, generator=g) * scale).to(DEV)


@pytest.mark.parametrize("m,widths,dtype", [(1, (128,), BF), (129, (256, 128), HF), (5003, (512, 128, 128), BF), (70000, (384, 128, 256), BF),
                                            (256, (128,) * 8, BF), (6144, (2048, 512, 512), BF)])
def test_quantize_side_and_join(m, widths, dtype):
    from kohakuwullm_amd.kernels.mxfp8.quantize import activation_matrix, join_codes, quantize_side, quantize_tokens

    xs = [_randn(m, w + 8 * j).to(dtype)[:, :w] for j, w in enumerate(widths)]  # pitches of their own
    whole = torch.cat(xs, 1)
    got = quantize_side([activation_matrix(x, dtype) for x in xs])
    for a, b in zip(got, quantize_tokens(whole, dtype)):
        assert a.shape == b.shape and torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    parts = [quantize_tokens(x.contiguous(), dtype)[:2] for x in xs]
    for a, b in zip(join_codes(parts), got[:2]):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))


def _layers(dtype, widths=(512, 128, 128), inp=256):
    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear

    torch.manual_seed(SEED)
    return torch.nn.ModuleList(MXFP8Linear(inp, w, dtype=dtype) for w in widths).to(DEV)


@pytest.mark.parametrize("shape,dtype,autocast,widths,silent", [
    ((1, 256), BF, None, (512, 128, 128), ()), ((700, 256), HF, None, (128, 256), ()), ((2, 65, 256), F32, BF, (512, 128, 128), ()),
    ((4096, 256), BF, None, (512, 128, 128), ()), ((300, 256), F32, HF, (512, 128, 128), (1,)), ((300, 256), BF, None, (128, 128, 128), (0, 2)),
])
def test_group_equals_the_layers(oracle, shape, dtype, autocast, widths, silent):
    from kohakuwullm_amd.kernels.mxfp8.linear import mxfp8_linear_group

    layers = _layers(dtype, widths)

    def step(run):
        x = _randn(*shape).to(dtype).requires_grad_(True)
        with torch.autocast("cuda", dtype=autocast or BF, enabled=autocast is not None):
            outs = run(x)
        picked = [j for j in range(len(widths)) if j not in silent]  # the others' results have no gradient
        dys = [_randn(shape[-2] + 7 * j, widths[j], scale=1e-2)[: shape[-2]].to(outs[j].dtype).expand_as(outs[j]) for j in picked]
        grads = torch.autograd.grad([outs[j] for j in picked], [x, *(layer.weight for layer in layers)], dys, allow_unused=True)
        return [*outs, *grads[1:]], grads[0]

    group, gdx = step(lambda x: mxfp8_linear_group(x, layers))
    alone, adx = step(lambda x: [layer(x) for layer in layers])
    for a, b in zip(group, alone):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape
            assert oracle.rel_error(a.detach().double().cpu(), b.detach().double().cpu()) < (1e-5 if a.dtype == F32 else 1e-3)
    assert gdx.dtype == adx.dtype and gdx.shape == adx.shape
    assert oracle.rel_error(gdx.double().cpu(), adx.double().cpu()) < (1e-5 if dtype == F32 else 4.6e-3)


def test_group_calls():
    from kohakuwullm_amd.kernels.mxfp8.linear import mxfp8_linear_group

    layers = _layers(BF)
    x = _randn(2, 50, 256).to(BF).requires_grad_(True)
    want = [y.detach().clone() for y in mxfp8_linear_group(x, layers)]
    with torch.no_grad():
        assert all(torch.equal(a, b) for a, b in zip(mxfp8_linear_group(x, layers), want))
    outs = mxfp8_linear_group(x, layers)
    outs[0].mul_(2.0)  # results may be written in place, as a single layer's may
    assert torch.equal(outs[0], want[0] * 2)
    # one weight's gradient alone
    (dw,) = torch.autograd.grad(mxfp8_linear_group(x, layers)[1].sum(), [layers[1].weight])
    (ref,) = torch.autograd.grad(layers[1](x).sum(), [layers[1].weight])
    assert torch.equal(dw, ref)
    # layer by layer: fp32 compute, no rows, a hook, a frozen weight (but not without gradients), padded widths, CPU inputs
    assert mxfp8_linear_group(x.float(), layers) is None and mxfp8_linear_group(x[:, :0], layers) is None
    handle = layers[2].register_forward_hook(lambda *a: None)
    assert mxfp8_linear_group(x, layers) is None
    handle.remove()
    layers[0].weight.requires_grad_(False)
    assert mxfp8_linear_group(x, layers) is None
    with torch.no_grad():
        assert mxfp8_linear_group(x, layers) is not None
    assert mxfp8_linear_group(x, _layers(BF, (200, 128))) is None and mxfp8_linear_group(x.cpu(), layers) is None
    assert mxfp8_linear_group(x, [torch.nn.Linear(256, 128)] * 2) is None
