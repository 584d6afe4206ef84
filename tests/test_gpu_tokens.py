"""The activation quantizers for any row count: every byte equals casting, padding with zero rows and columns and the
row + column quantizer (or the SwiGLU ones) on the padded matrix, at the edges of their tiles and of the token extent."""

import pytest
import torch
import torch.nn.functional as F

from conftest import SEED

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _u8(t):
    return t.view(torch.uint8).cpu()


def _draw(*shape, dtype=BF, scale=1.0):
    g = torch.Generator().manual_seed(SEED + shape[0])
    return (torch.randn(*shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("m,kv,k,dtype,compute", [
    (1, 32, 32, BF, BF), (31, 128, 128, HF, HF), (33, 104, 128, BF, BF), (128, 256, 256, F32, F32), (129, 1000, 1024, BF, BF),
    (700, 160, 160, F32, BF), (1535, 256, 256, F32, HF), (5003, 512, 512, BF, BF), (70000, 1536, 1536, HF, HF),
    # whole tiles, whose kernels test nothing: a few of them (kept as loaded) and more than eight per CU; four and a half
    # per CU, which are tested all the same
    (512, 384, 384, HF, HF), (16384, 2176, 2176, BF, BF), (9216, 2048, 2048, HF, HF), (6144, 3072, 3072, BF, BF),
])
def test_quantize_tokens(oracle, m, kv, k, dtype, compute):
    from kohakuwullm_amd.kernels.mxfp8.quantize import activation_matrix, quantize_tokens, rows_of_stage_major, token_extent

    x = _draw(m, kv, dtype=dtype)
    q, s, qt, st = quantize_tokens(activation_matrix(x.to(DEV), compute), compute, k)
    mt = token_extent(m)
    assert mt % 128 == 0 and m <= mt < m + 128 + m / 16 + 128 and qt.shape == (mt // 128, k, 128) and st.shape == (k, mt // 32)
    if k == kv:  # the row axis alone, from a pitched view too
        for src in (x.to(DEV), F.pad(x, (0, 16)).to(DEV)[:, :kv]):
            q1, s1, qt1, st1 = quantize_tokens(activation_matrix(src, compute), compute, token_axis=False)
            assert qt1 is None and st1 is None and torch.equal(_u8(q1), _u8(q)) and torch.equal(s1, s)
    padded = F.pad(x.to(compute), (0, k - kv, 0, mt - m))
    rq, rs = oracle.quantize_rows(padded[:m])
    cq, cs = oracle.quantize_cols(padded)
    assert torch.equal(_u8(q), rq) and torch.equal(s.cpu(), rs)
    assert torch.equal(_u8(rows_of_stage_major(qt)), cq) and torch.equal(st.cpu(), cs)


@pytest.mark.parametrize("m,h,dtype", [(1, 128, BF), (129, 256, HF), (1500, 384, BF), (160, 128, BF)])
def test_swiglu_tokens(oracle, m, h, dtype):
    """Unrounded: the bytes of the fixed-shape kernels on zero-padded inputs.  Rounded: the casts of what PyTorch's 16-bit
    operators and their autograd give on the CPU, up to ties (its sigmoid is libm's, here the hardware exponential's)."""
    from kohakuwullm_amd.kernels.mxfp8.mlp import swiglu_bwd_mx_dual, swiglu_bwd_tokens, swiglu_mx_dual, swiglu_tokens
    from kohakuwullm_amd.kernels.mxfp8.quantize import rows_of_stage_major, token_extent

    gu, dh = _draw(m, 2 * h, dtype=dtype, scale=1.5), _draw(m, h, dtype=dtype, scale=1e-2)
    mt = token_extent(m)
    guz, dhz = F.pad(gu, (0, 0, 0, mt - m)).to(DEV), F.pad(dh, (0, 0, 0, mt - m)).to(DEV)
    for got, want in ((swiglu_tokens(gu.to(DEV)), swiglu_mx_dual(guz)), (swiglu_bwd_tokens(dh.to(DEV), gu.to(DEV)), swiglu_bwd_mx_dual(dhz, guz))):
        q = got[0] if got[0].dim() == 2 else rows_of_stage_major(got[0])
        assert torch.equal(_u8(q), _u8(want[0][:m])) and torch.equal(got[1], want[1][:m])
        assert torch.equal(_u8(rows_of_stage_major(got[2])), _u8(want[2])) and torch.equal(got[3], want[3])
    for rounded in (False, True):
        both, one = swiglu_tokens(gu.to(DEV), rounded), swiglu_tokens(gu.to(DEV), rounded, token_axis=False)
        assert torch.equal(_u8(one[0]), _u8(both[0])) and torch.equal(one[1], both[1]) and one[2] is None and one[3] is None

    gc = gu.clone().requires_grad_(True)
    gate, up = gc.chunk(2, dim=-1)
    hc = F.silu(gate) * up
    hc.backward(dh)
    for got, ref in ((swiglu_tokens(gu.to(DEV), rounded=True), hc.detach()), (swiglu_bwd_tokens(dh.to(DEV), gu.to(DEV), rounded=True), gc.grad)):
        q = got[0] if got[0].dim() == 2 else rows_of_stage_major(got[0])
        for codes, scales, want in ((q, got[1], ref), (rows_of_stage_major(got[2]), got[3], F.pad(ref, (0, 0, 0, mt - m)).t().contiguous())):
            # a 16-bit intermediate that rounds the other way moves a value by one 16-bit ulp, 1/32 (bf16) or 1/256 of an
            # e4m3 step, so at most that share of the values next to a boundary could differ; few intermediates do
            wq, ws = oracle.quantize_rows(want)
            assert (_u8(codes) != wq).float().mean() < 1e-3 and (scales.cpu() != ws).float().mean() < 1e-3
            assert oracle.rel_error(oracle.dequant(_u8(codes), scales.cpu()), oracle.dequant(wq, ws)) < 2e-3
