"""Activations as programs hold them -- views at odd offsets of flat buffers, slices, broadcast rows -- through the entry points
whose quantizers fetch 16 bytes at a time: the host's repair on the CPU, the modules on the GPU."""

import pytest
import torch

from conftest import SEED

DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _views(m, k, dtype, device="cpu"):
    """Tensors of shape (m, k) and one content each, in layouts the kernels do not take as they are."""
    g = torch.Generator().manual_seed(SEED)
    flat = torch.randn(m * k + 8, generator=g).to(dtype).to(device)
    wide = torch.randn(m, k + 4, generator=g).to(dtype).to(device)
    return {
        "offset": flat[4 : 4 + m * k].view(m, k), "odd offset": flat[1 : 1 + m * k].view(m, k), "pitch": wide[:, :k],
        "broadcast": flat[:k].expand(m, k), "transposed": flat[: m * k].view(k, m).t(), "one row": wide[:1, :k],
    }


@pytest.mark.parametrize("compute,dtype", [(BF, BF), (HF, HF), (BF, F32), (F32, F32)])
@pytest.mark.parametrize("m", [1, 3, 128])
def test_activation_matrix_is_what_the_kernels_take(m, compute, dtype):
    from kohakuwullm_amd.kernels.mxfp8.quantize import activation_matrix

    for name, x in _views(m, 64, dtype).items():
        got = activation_matrix(x, compute)
        assert torch.equal(got, x), name
        assert got.stride(1) == 1 and got.stride(0) >= 64 and got.stride(0) * got.element_size() % 16 == 0 and got.data_ptr() % 16 == 0, name
    fine = torch.zeros(m, 80, dtype=compute)[:, :64]
    assert activation_matrix(fine, compute).data_ptr() == fine.data_ptr()  # and is not copied


def _modules(dtype):
    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear, mxfp8_linear_group
    from kohakuwullm_amd.models.mlp import MXFP8SwiGLU, SwiGLU
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    torch.manual_seed(SEED)
    swapped = SwiGLU(256, hidden=384).to(DEV).to(dtype)
    swap_mxfp8(swapped)
    layers = torch.nn.ModuleList(MXFP8Linear(256, w) for w in (256, 128)).to(DEV).to(dtype)
    group = torch.nn.Module()
    group.layers = layers
    group.forward = lambda x: torch.cat(mxfp8_linear_group(x, layers), -1)
    return {"linear": MXFP8Linear(256, 384).to(DEV).to(dtype), "linear, width % 8": MXFP8Linear(256, 100).to(DEV).to(dtype), "group": group,
            "swapped": swapped, "fused": MXFP8SwiGLU(256, hidden=384).to(DEV).to(dtype)}


def _step(module, x, dy, autocast):
    for p in module.parameters():
        p.grad = None
    x = x.detach().requires_grad_(True)
    with torch.autocast("cuda", dtype=BF, enabled=autocast):
        y = module(x)
        with torch.no_grad():
            alone = module(x)
    y.backward(dy.to(y.dtype))
    return [y.detach(), alone, x.grad, *(p.grad for p in module.parameters())]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,autocast", [(BF, False), (HF, False), (F32, True)])
@pytest.mark.parametrize("m", [1, 129, 256])
def test_modules_take_any_layout(m, dtype, autocast):
    for label, module in _modules(dtype).items():
        for name, x in _views(m, 256, dtype, DEV).items():
            if name == "one row" and m > 1:
                continue
            with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=autocast):
                width = module(x).shape[1]
            plain = (torch.randn(m, width, device=DEV) * 1e-2).to(BF if autocast else dtype)
            flat = torch.cat((plain.new_zeros(4), plain.reshape(-1)))
            want = _step(module, x.contiguous().clone(), plain, autocast)
            for dy in (plain, flat[4:].view(m, width)):  # (autograd leaves a gradient's layout alone)
                for a, b in zip(_step(module, x, dy, autocast), want):
                    assert a.dtype == b.dtype and torch.equal(a, b), (label, name)
        # a gradient that is one row for every token, as a sum over the tokens gives it
        x = torch.randn(m, 256, device=DEV).to(dtype)
        row = plain[:1].expand(m, width)
        for a, b in zip(_step(module, x, row, autocast), _step(module, x, row.clone(memory_format=torch.contiguous_format), autocast)):
            assert torch.equal(a, b), label


@pytest.mark.parametrize("m,k,entry", [
    (65535 * 128, 2048, "mx_quantize_tokens"), (65535 * 128 + 1, 1024, "mx_quantize_tokens"),
    (65535 * 128 + 1, 2080, "mx_quantize_rows"), (2**25, 512, "mx_quantize_rows"),
])
def test_forwards_past_the_tile_and_row_kernels_take_the_general_one(monkeypatch, m, k, entry):
    from kohakuwullm_amd.kernels.mxfp8 import quantize

    calls = []
    monkeypatch.setattr(quantize._lib, "require_gpu", lambda *a: None)
    monkeypatch.setattr(quantize._lib, "invoke", lambda name, work, x, *a: calls.append((name, x.dtype)))
    x = torch.empty(m, k, dtype=F32, device="meta")
    q, s, qt, st = quantize.quantize_tokens(x, BF, token_axis=False)
    assert calls == [(entry, BF if entry == "mx_quantize_rows" else F32)]  # rounded in front of it, as a cast would
    assert q.shape == (m, k) and s.shape == (m, k // 32) and (qt is None) == (st is None)


def test_token_extent_stays_within_the_tile_kernels_grid():
    from kohakuwullm_amd.kernels.mxfp8.quantize import TILE_ROWS, token_extent

    assert token_extent(TILE_ROWS) == TILE_ROWS and token_extent(TILE_ROWS - 128) <= TILE_ROWS
    assert token_extent(5024) == 5120 and token_extent(2176) == 2176


@pytest.mark.gpu
def test_swapped_block_past_the_tile_kernels(tokens=65535 * 128 + 1):
    """Frozen weights, more tokens than a token-axis quantizer covers: forward and dX, row by row as in a short batch."""
    from kohakuwullm_amd.models.mlp import SwiGLU
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    torch.manual_seed(SEED)
    block = SwiGLU(128, hidden=128).to(DEV).to(BF)
    swap_mxfp8(block)
    block.requires_grad_(False)
    tail = torch.randn(256, 128, device=DEV).to(BF)
    x = tail.repeat(-(-tokens // 256) + 1, 1)[-tokens:]
    out = []
    for part in (x, tail):
        part = part.detach().requires_grad_(True)
        y = block(part)
        y.backward(y.detach())
        out.append((y.detach()[-256:].clone(), part.grad[-256:].clone()))
    for a, b in zip(*out):
        assert torch.equal(a, b)


def _off(t):
    """A copy of ``t`` one element past an allocation's start, as an arena of a saved-tensor hook may give it back."""
    return t.new_empty(t.numel() + 1)[1:].view(t.shape).copy_(t)


def test_saved_operands_at_odd_offsets_are_laid_back(monkeypatch):
    """What reaches the kernels that take aligned operands alone: stage-major codes, joined weights, the saved projection."""
    import ctypes

    from kohakuwullm_amd import _lib
    from kohakuwullm_amd.kernels.mxfp8 import mlp, quantize

    seen = {}
    monkeypatch.setattr(_lib, "require_gpu", lambda *a: None)
    monkeypatch.setattr(_lib, "gemm_workspace", lambda t: torch.empty(1))
    monkeypatch.setattr(_lib, "invoke", lambda name, work, like, *args: seen.__setitem__(name, (args, _records(name, args))))

    def _records(name, args):
        record = {"mx_join_codes": _lib.CodeSource, "mx_gemm_nt_batch": _lib.GemmProblem}.get(name)
        if record is None:
            return None
        at = args[0] if isinstance(args[0], int) else ctypes.addressof(args[0]._obj)
        return [{n: getattr(r, n) for n, _ in record._fields_} for r in (record * args[1]).from_buffer_copy(ctypes.string_at(at, ctypes.sizeof(record) * args[1]))]

    f8, u8 = torch.float8_e4m3fn, torch.uint8
    codes, scales = torch.zeros(256, 128).to(f8), torch.zeros(256, 4, dtype=u8)
    quantize.join_codes([(_off(codes), _off(scales)), (codes, scales)])
    for r in seen["mx_join_codes"][1]:
        assert r["codes"] % 16 == 0 and r["ld"] == 128 and r["scales"] % 4 == 0 and r["lds"] == 4
    panels = codes.view(2, 128, 128)
    s8 = torch.zeros(128, 8, dtype=u8)
    quantize.mxfp8_matmul_pq_batch([(_off(panels), s8, _off(panels), s8), (panels, s8, _off(codes.view(128, 256)), s8)])
    for r in seen["mx_gemm_nt_batch"][1]:
        assert r["aq"] % 16 == 0 and r["bq"] % 16 == 0
    mlp.swiglu_bwd_tokens(torch.zeros(5, 128, dtype=BF), _off(torch.zeros(5, 256, dtype=BF)))
    assert seen["mx_swiglu_bwd_quantize_tokens"][0][2] % 16 == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,autocast", [(BF, False), (F32, True)])
def test_modules_under_a_saved_tensor_hook(dtype, autocast):
    for label, module in _modules(dtype).items():
        x = torch.randn(129, 256, device=DEV).to(dtype)
        with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=autocast):
            dy = torch.randn_like(module(x)) * 1e-2
        want = _step(module, x, dy, autocast)
        with torch.autograd.graph.saved_tensors_hooks(_off, lambda t: t):
            got = _step(module, x, dy, autocast)
        for a, b in zip(got, want):
            # products of row-major weights at odd offsets run on the element-wise kernel: fp32 sums in another order, and a
            # 16-bit result rounded the other way is off by 2^-8 of itself at most
            assert a.dtype == b.dtype and float((a - b).float().norm()) <= 4e-3 * float(b.float().norm()), label
