"""The small-tile GEMM (csrc/mx_gemm_ring.h) and the one for few rows (csrc/mx_gemm_skinny.h) against dequantize-then-matmul in
fp64 at the edges of what they take: single groups of four K stages, ragged and single rows, K slices, padded rows, stage-major
operands, several products in a launch.

Tolerances are those of the other GEMM tests: 1e-4 in fp32 (the block-scaled MFMA's own adder), 4e-3 in bf16 (its rounding)."""

import pytest
import torch

from conftest import SEED

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F8 = torch.float8_e4m3fn
TOL = {torch.float32: 1e-4, torch.bfloat16: 4e-3, torch.float16: 6e-4}


def _operands(oracle, m, n, k):
    g = torch.Generator().manual_seed(SEED + m)
    a = (torch.randn(m, k, generator=g)).bfloat16()
    b = (torch.randn(n, k, generator=g) * 0.02).bfloat16()
    return *oracle.quantize_rows(a), *oracle.quantize_rows(b)


def _dev(ops, panels=False):
    aq, a_s, bq, b_s = (t.to(DEV) for t in ops)
    if panels:
        aq, bq = (t.view(t.shape[0], t.shape[1] // 128, 128).permute(1, 0, 2).contiguous() for t in (aq, bq))
    return aq.view(F8), a_s, bq.view(F8), b_s


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 512), (1, 3072, 2048), (127, 129, 512), (128, 128, 1024), (129, 257, 1536), (700, 260, 4096),
    (300, 520, 8192),  # 15 tiles, cut into eight K slices
    (16, 40, 16384), (130, 1000, 10240),  # slices of unequal length
    # the shapes above with up to 128 rows go to the kernel for few rows; these of their kind do not
    (129, 1, 512), (129, 3072, 2048), (255, 129, 512), (256, 128, 1024), (129, 40, 16384), (100, 1000, 10240), (128, 5000, 512),
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_ring_gemm(oracle, m, n, k, dtype):
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq

    ops = _operands(oracle, m, n, k)
    ref = oracle.gemm_nt(*ops)
    out = mxfp8_matmul_pq(*_dev(ops), dtype)
    assert oracle.rel_error(out.cpu(), ref) < TOL[dtype]
    padded = mxfp8_matmul_pq(*_dev(ops), dtype, out_pad=24)
    assert padded.stride(0) == n + 24 and torch.equal(padded, out)
    assert torch.equal(mxfp8_matmul_pq(*_dev(ops, panels=True), dtype), out)


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 128), (1, 17, 384), (15, 16, 640), (16, 4100, 1024), (17, 48, 1152), (32, 4112, 2048), (33, 200, 896), (64, 520, 4224), (64, 4128, 256),
    (65, 72, 1280), (128, 129, 2176),  # the last group of 16 rows and of 16 columns, one K stage per wave, none, several
    (7, 4112, 4096), (16, 4112, 4352), (16, 300, 3200),  # up to 16 rows: one stage at a time on a full chip, two past four stages, two
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_gemm_of_few_rows(oracle, m, n, k, dtype):
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, mxfp8_matmul_pq_batch

    ops = _operands(oracle, m, n, k)
    out = mxfp8_matmul_pq(*_dev(ops), dtype)
    assert oracle.rel_error(out.cpu(), oracle.gemm_nt(*ops)) < TOL[dtype]
    padded = mxfp8_matmul_pq(*_dev(ops), dtype, out_pad=3)
    assert padded.stride(0) == n + 3 and torch.equal(padded, out)
    assert torch.equal(mxfp8_matmul_pq(*_dev(ops, panels=True), dtype), out)
    other = _operands(oracle, 9, 50, 512)  # beside a product with fewer rows and another K: the same sums
    both = mxfp8_matmul_pq_batch([_dev(ops), _dev(other)], dtype)
    assert torch.equal(both[0], out) and oracle.rel_error(both[1].cpu(), oracle.gemm_nt(*other)) < TOL[dtype]


@pytest.mark.parametrize("m,n,k", [
    (130, 300, 128), (257, 129, 256), (200, 264, 384),  # without a whole group
    (129, 1, 640), (129, 130, 768), (300, 40, 1408), (513, 260, 2176), (300, 257, 896), (256, 128, 1152),
    (129, 40, 8320), (130, 200, 16384 + 384),  # K slices whose last one ends inside a group
    (130, 200, 14464), (130, 200, 14592), (130, 200, 14720),  # ... or is one to three stages alone
])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ring_gemm_ends_inside_a_group(oracle, m, n, k, dtype):
    """One to three stages in the last group, or in all; the matrices end where their allocations do."""
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq

    ops = _operands(oracle, m, n, k)
    out = mxfp8_matmul_pq(*_dev(ops), dtype)
    assert oracle.rel_error(out.cpu(), oracle.gemm_nt(*ops)) < TOL[dtype]
    assert torch.equal(mxfp8_matmul_pq(*_dev(ops, panels=True), dtype), out)


def test_ring_gemm_several_products_in_one_launch(oracle):
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, mxfp8_matmul_pq_batch

    shapes = [(515, 256, 512), (64, 384, 8192), (1, 129, 1024), (256, 512, 8192), (300, 40, 2048)]
    ops = [_operands(oracle, *s) for s in shapes]
    problems = [_dev(o, panels=i % 2 == 1) for i, o in enumerate(ops)]
    outs = mxfp8_matmul_pq_batch(problems, torch.float32)
    for o, p, out in zip(ops, problems, outs):
        assert oracle.rel_error(out.cpu(), oracle.gemm_nt(*o)) < 1e-4
        alone = mxfp8_matmul_pq(*p, torch.float32)
        assert oracle.rel_error(out.cpu(), alone.double().cpu()) < 1e-5  # the same sums, K slices apart


def test_ring_gemm_short_and_long_products_in_one_launch(oracle):
    """The gradients of a layer over few tokens: dX over the outputs beside dW over one to three panels."""
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq_batch

    ops = [_operands(oracle, *s) for s in [(200, 512, 1536), (1536, 512, 256), (130, 60, 640), (264, 129, 384)]]
    for o, out in zip(ops, mxfp8_matmul_pq_batch([_dev(o, panels=i == 1) for i, o in enumerate(ops)], torch.bfloat16)):
        assert oracle.rel_error(out.cpu(), oracle.gemm_nt(*o)) < TOL[torch.bfloat16]


@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (3, 17, 640), (16, 4100, 4096), (17, 48, 1152), (32, 520, 2048)])
@pytest.mark.parametrize("xt,ct", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16), (torch.float32, torch.bfloat16), (torch.float32, torch.float16)])
def test_activations_quantized_inside_the_product(m, n, k, xt, ct):
    """The bits of the row quantizer and the product behind it, for rows at any pitch; zeros, infinities and NaN among them."""
    import ctypes

    from kohakuwullm_amd import _lib
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, quantize_mx

    g = torch.Generator(device=DEV).manual_seed(SEED + m)
    x = torch.randn(m, k + 8, device=DEV, generator=g).to(xt)[:, :k]
    x[0, :32] = 0
    x[-1, 40], x[-1, 70] = float("inf"), float("nan")
    ws = [quantize_mx(torch.randn(c, k, device=DEV, generator=g).bfloat16()) for c in (n, 50)]
    outs = [torch.empty(m, w[0].shape[0], device=DEV, dtype=ct) for w in ws]

    def call(rows=m, depth=k, out=ct, at=0):
        records = _lib.words(_lib.GemmProblem, [(0, 0, q.data_ptr(), s.data_ptr(), o.data_ptr(), rows, q.shape[0], depth, 0, 0, k, k // 32, q.shape[0])
                                                for (q, s), o in zip(ws, outs)])
        return _lib.load().mx_activation_gemm_nt(x.data_ptr() + at, _lib.MX_DTYPE[xt], x.stride(0), ctypes.byref(records), 2, _lib.MX_DTYPE[out], _lib.stream_of(x))

    assert call() == _lib.MX_OK
    xq, xs = quantize_mx(x.to(ct))
    for o, w in zip(outs, ws):
        want = mxfp8_matmul_pq(xq, xs, *w, ct)
        assert torch.equal(o.view(torch.int16), want.view(torch.int16)) or torch.equal(o.isnan(), want.isnan()) and torch.equal(o.nan_to_num(), want.nan_to_num())
    refused = [call(rows=33), call(depth=k - 32), call(at=2), call(out=torch.float32)]
    assert refused == [_lib.MX_EUNSUPPORTED] * 4


@pytest.mark.parametrize("rows,depth,columns,count,taken", [
    (16, 4096, 64, 1, True), (16, 4224, 64, 1, False), (17, 2048, 64, 1, True), (17, 2176, 64, 1, False), (32, 128, 64, 1, True), (33, 128, 64, 1, False),
    (17, 256, 4096, 1, True), (17, 256, 4112, 1, False), (17, 256, 2048, 2, True), (17, 256, 2064, 2, False), (16, 256, 20000, 1, True),
    (8, 256, 64, 4, True), (8, 256, 64, 5, False),
])
def test_which_activations_are_quantized_inside_the_product(rows, depth, columns, count, taken):
    """The limits that the header states (256 CUs), and nothing written past them."""
    import ctypes

    from kohakuwullm_amd import _lib
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, quantize_mx

    g = torch.Generator(device=DEV).manual_seed(SEED)
    x = torch.randn(rows, depth, device=DEV, generator=g).bfloat16()
    q, s = quantize_mx(torch.randn(columns, depth, device=DEV, generator=g).bfloat16())
    out = torch.full((count, rows, columns), 3.0, device=DEV, dtype=torch.bfloat16)
    records = _lib.words(_lib.GemmProblem, [(0, 0, q.data_ptr(), s.data_ptr(), o.data_ptr(), rows, columns, depth, 0, 0, depth, depth // 32, columns) for o in out])
    status = _lib.load().mx_activation_gemm_nt(x.data_ptr(), 0, depth, ctypes.byref(records), count, 0, _lib.stream_of(x))
    assert status == (_lib.MX_OK if taken else _lib.MX_EUNSUPPORTED)
    want = mxfp8_matmul_pq(*quantize_mx(x), q, s, torch.bfloat16) if taken else torch.full_like(out[0], 3.0)
    assert all(_close(o, want) for o in out)


def _close(a, b):
    return ((a.double() - b.double()).norm() <= 4e-3 * b.double().norm()).item()  # the products' sums may be cut differently


@pytest.mark.parametrize("k", [(8192, 8192), (8320, 8192), (8192 + 32, 9216)])  # 16 scale bytes, 4 and 1 at a time; slices of unequal length
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_batch_cuts_the_tiles_of_its_last_round(k, dtype):
    """130 tiles each on half of the chip: a round of whole tiles and two tiles in K slices, ragged rows and columns among them."""
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq_batch

    g = torch.Generator(DEV).manual_seed(SEED)

    def codes(rows, cols):  # every finite code, scales over eight octaves
        q = torch.randint(0, 254, (rows, cols), generator=g, device=DEV, dtype=torch.uint8)
        q = q + (q >= 127).to(torch.uint8)
        return q, torch.randint(115, 123, (rows, cols // 32), generator=g, device=DEV, dtype=torch.uint8)

    def value(q, s):
        return q.view(F8).double() * torch.exp2(s.double() - 127.0).repeat_interleave(32, dim=1)

    problems = [(*codes(m, kk), *codes(n, kk)) for (m, n), kk in zip(((3300, 2500), (2490, 3310)), k)]
    for (aq, a_s, bq, b_s), out in zip(problems, mxfp8_matmul_pq_batch([(a.view(F8), s, b.view(F8), t) for a, s, b, t in problems], dtype)):
        ref = value(aq, a_s) @ value(bq, b_s).T
        assert ((out.double() - ref).norm() / ref.norm()).item() < TOL[dtype]


def _sums(m, n, k):
    """Operands whose product shows in which order fp32 sums took its K stages: 2^24 from the first of them, in which later ones
    are lost, and 1 from every other."""
    a, b = torch.zeros(m, k, dtype=torch.uint8), torch.zeros(n, k, dtype=torch.uint8)
    a[:, ::128], b[:, ::128] = 0x38, 0x38  # one 1.0 per stage
    a_s, b_s = torch.full((m, k // 32), 127, dtype=torch.uint8), torch.full((n, k // 32), 127, dtype=torch.uint8)
    b_s[:, 0] = 127 + 24
    return a, a_s, b, b_s


@pytest.mark.parametrize("m,n,k,order", [
    # eighths of K and their sums in order: the kernel for few rows
    (16, 4096, 28672, "eighths"), (16, 16384, 1536, "eighths"), (64, 2048, 4096, "eighths"), (128, 2048, 4096, "eighths"), (32, 4096, 4096, "eighths"),
    # a long K, whose eighths are walks of many stages: ring tiles in four slices of whole groups
    (64, 8192, 8192, "quarters"), (128, 512, 8192, "quarters"), (48, 5000, 12800, "quarters"),
    # many columns, whose workgroups share the CUs: ring tiles, or 256 x 256 ones past four rounds of them
    (64, 32768, 1536, "whole"), (32, 49152, 1536, "whole"), (128, 5120, 1536, "whole"), (64, 150000, 512, "whole"),
])
def test_few_rows_go_where_their_columns_and_depth_say(m, n, k, order):
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq

    ops = _dev(_sums(m, n, k))
    out = mxfp8_matmul_pq(*ops, torch.float32)
    stages = k // 128
    per = {"eighths": -(-stages // 8), "quarters": (-(-stages // 4) + 3) // 4 * 4, "whole": stages}[order]
    assert torch.equal(out, torch.full_like(out, 2.0**24 + stages - per))


def test_few_rows_in_a_batch_share_the_choice():
    """Columns of all products together: 8192 each are few enough alone, four times 8192 are not."""
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, mxfp8_matmul_pq_batch

    ops = _dev(_sums(64, 8192, 1536))
    assert (mxfp8_matmul_pq(*ops, torch.float32) == 2.0**24 + 10).all()
    for out in mxfp8_matmul_pq_batch([ops] * 4, torch.float32):
        assert (out == 2.0**24).all()


def test_few_rows_without_scratch_keep_a_long_k():
    """A caller without a workspace gets no K slices from the other kernels, so the few-row kernel's eighths are the quicker ones."""
    from kohakuwullm_amd import _lib

    aq, a_s, bq, b_s = _dev(_sums(64, 512, 8192))
    out = torch.empty(64, 512, device=DEV)
    call = lambda ws, n: _lib.load().mx_gemm_nt(aq.data_ptr(), a_s.data_ptr(), bq.data_ptr(), b_s.data_ptr(), out.data_ptr(), 2, 64, 512, 8192, 8192, 256,
                                                8192, 256, 512, 0, ws, n, _lib.stream_of(aq))  # noqa: E731
    assert call(0, 0) == _lib.MX_OK and (out == 2.0**24 + 56).all()
