"""The C++ host path (csrc/mx_host.cpp) against the Python one it stands for: the same launches, so the same bits, for every
layout, type and option a call may have; and what it leaves to Python, told by a None with nothing launched."""

import contextlib

import pytest
import torch

from conftest import SEED

DEV = "cuda:0"
BF, F16, F32 = torch.bfloat16, torch.float16, torch.float32


class _Own(torch.Tensor):
    pass


def test_calls_that_are_not_plain_are_declined():
    from torch.utils._python_dispatch import TorchDispatchMode

    from kohakuwullm_amd import host

    x, w = torch.zeros(32, 128, dtype=BF), torch.zeros(64, 128, dtype=torch.uint8)
    s = torch.zeros(64, 4, dtype=torch.uint8)
    calls = [
        lambda t: host.quantize_rows(t), lambda t: host.quantize_tokens(t, BF, 0, True), lambda t: host.quantize_side([t, t]),
        lambda t: host.join_codes([(w, s), (w, s)]), lambda t: host.quantize_dual_batch([t]), lambda t: host.matmul(w, s, w, s, BF, 0),
        lambda t: host.matmul_batch([(w, s, w, s)], BF), lambda t: host.linear_eval(t, t, w, s), lambda t: host.linear_forward(t, BF, w, s, True),
        lambda t: host.group_forward(t, BF, [(w, s, w, s)] * 2, True), lambda t: host.rmsnorm_forward(t, None, 1e-6),
        lambda t: host.route_forward(t, t, None, 2, True, 1.0, True), lambda t: host.quantize_rows(None), lambda t: host.quantize_rows(3),
        lambda t: host.matmul(w, s, w, s, "bf16", 0),
    ]
    for t in (x, x.as_subclass(_Own), torch.nn.Parameter(x), x.to("meta"), torch.zeros(0, 128, dtype=BF)):
        for i, call in enumerate(calls):
            assert call(t) is None, (i, type(t), t.device)
    with torch.no_grad():
        assert not host.unrecorded(x) and not host.unrecorded(3)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        assert calls[0](x) is None


def test_sizes_and_limits_are_those_of_the_python_functions():
    from kohakuwullm_amd import _host
    from kohakuwullm_amd.kernels.mxfp8 import grouped, quantize

    assert _host.constants == {n: getattr(grouped if n == "SCALE_ROW_SLACK" else quantize, n) for n in _host.constants} and len(_host.constants) == 5
    assert grouped.WGRAD_ROW_TILE == quantize.PANEL and grouped.TOKEN_PITCH_PAD == 0
    for rows in (1, 31, 128, 129, 511, 513, 2048, 2049, 8065, 16384, 65535 * 128 - 1, 65535 * 128, 65535 * 128 + 1, 2**40 + 7):
        for experts in (1, 64):
            assert _host.extents(rows, rows, experts) == (quantize.token_extent(rows), grouped.padded_rows(rows, experts))


def test_first_use_with_another_library_or_binding_installed():
    """Whatever stands in the binding when the extension is first used, it makes calls for the product library and the binding's own
    ``invoke`` alone."""
    import subprocess
    import sys

    code = """
from kohakuwullm_amd import _lib, host
own, _lib.invoke = _lib.invoke, lambda *a: None
with _lib.variants_library():
    inside = [host.engaged()]
    _lib.invoke = own
    inside.append(host.engaged())
assert inside == [False, False], inside
assert host.engaged()
_lib.TIMER = []
assert not host.engaged()
"""
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300)


@pytest.mark.parametrize("spoil", ["sys.modules['kohakuwullm_amd._host'] = None", "torch.__version__ = '1.0.0'"])
def test_without_the_extension_every_call_takes_the_python_way(spoil):
    """Not built, or built against another PyTorch: a warning, and the functions in front of it do what they do for any other call."""
    import subprocess
    import sys

    code = f"""
import sys, warnings, torch
{spoil}
from kohakuwullm_amd import _lib, host
from kohakuwullm_amd.kernels.mxfp8 import quantize_mx
x = torch.zeros(32, 128)
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter('always')
    assert host.quantize_rows(x) is None and host.quantize_rows(x) is None and not host.unrecorded(x) and not host.engaged()
assert [w.category for w in seen] == [RuntimeWarning], seen
try:
    quantize_mx(x)
except _lib.MXFP8LibraryError as error:
    assert 'lives on cpu' in str(error)
else:
    raise AssertionError
"""
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300)


@contextlib.contextmanager
def _python():
    """Calls inside go the Python way: a timer is installed."""
    from kohakuwullm_amd import _lib

    _lib.TIMER = []
    try:
        yield
    finally:
        _lib.TIMER = None


def _bits(t):
    return t.contiguous().flatten().view(torch.uint8)


def _both(run):
    got = run()
    with _python():
        want = run()
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a is None) == (b is None), i
        if a is not None:
            assert a.shape == b.shape and a.dtype == b.dtype and a.stride() == b.stride() and torch.equal(_bits(a), _bits(b)), i


def _layouts(tokens, width, dtype):
    """The same values as they may lie: flat, batched, pitched, transposed, at an odd offset, broadcast over the batch."""
    g = torch.Generator(device=DEV).manual_seed(SEED)
    base = torch.randn(tokens, width, device=DEV, generator=g).to(dtype)
    odd = torch.empty(tokens * width + 1, device=DEV, dtype=dtype)[1:].view(tokens, width).copy_(base)
    pitched = torch.empty(tokens, width + 8, device=DEV, dtype=dtype)[:, :width].copy_(base)
    return {"flat": base, "batched": base.view(1, tokens, width), "odd": odd, "pitched": pitched, "transposed": base.t().contiguous().t(),
            "broadcast": base[:1].expand(3, tokens, width), "empty": base[:0]}


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["flat", "batched", "odd", "pitched", "transposed", "broadcast", "empty"])
@pytest.mark.parametrize("dtype,master,autocast", [(BF, BF, False), (F16, F16, False), (F32, F32, True), (BF, F32, False)])
@pytest.mark.parametrize("tokens,inp,out", [(1, 128, 1000), (33, 256, 384)])
def test_linear(layout, dtype, master, autocast, tokens, inp, out):
    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear

    torch.manual_seed(SEED)
    lin = MXFP8Linear(inp, out).to(DEV).to(master)
    x0 = _layouts(tokens, inp, dtype)[layout]

    def run(train=True, weight=True):
        lin.weight.requires_grad_(weight)
        lin.weight.grad = None
        x = x0.detach().requires_grad_(train)
        with torch.autocast("cuda", dtype=BF, enabled=autocast), torch.set_grad_enabled(train):
            y = lin(x)
        if not train:
            assert y.grad_fn is None
            return [y]
        y.backward(torch.ones_like(y).mul_(1e-2))
        return [y.detach(), x.grad, lin.weight.grad]

    _both(run)
    _both(lambda: run(True, False))
    _both(lambda: run(False))


@pytest.mark.gpu
@pytest.mark.parametrize("out,tensors", [(16384, 1), (16400, 3)])  # the result; codes and scale bytes of the rows as well
def test_rows_are_quantized_inside_the_product_up_to_64_columns_per_cu(out, tensors):
    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear

    torch.manual_seed(SEED)
    lin, x = MXFP8Linear(256, out).to(DEV).to(BF), torch.randn(16, 256, device=DEV).to(BF)
    with torch.no_grad():
        _both(lambda: [lin(x)])
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        lin(x)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == tensors


@pytest.mark.gpu
def test_calls_are_declined_in_front_of_the_first_launch():
    """A weight that only the product would object to: nothing has been allocated for the quantizer in front of it."""
    from kohakuwullm_amd import host
    from kohakuwullm_amd.kernels.mxfp8 import quantize_mx

    x = torch.randn(40, 256, device=DEV).to(BF)
    q, s = quantize_mx(torch.randn(512, 256, device=DEV).to(BF))
    q2, s2 = quantize_mx(torch.randn(256, 256, device=DEV).to(BF))
    bad = s.t().contiguous().t(), s[:-1], s.float()
    with torch.no_grad():
        assert host.linear_eval(x, x, q, s) is not None
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        for scale in bad:
            assert host.linear_forward(x, BF, q, scale, True) is None and host.linear_eval(x, x, q, scale) is None
            assert host.group_forward(x, BF, [(q, scale, q, scale)], True) is None
            assert host.swiglu_mlp_forward(x, BF, (q, scale), (q2, s2), False, False, False, 0) is None
            assert host.linear_backward(x, BF, None, None, q[:, :256], scale, True, False, BF, BF) is None
        assert torch.cuda.memory_stats()["allocation.all.allocated"] == before


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["flat", "batched", "pitched", "transposed"])
@pytest.mark.parametrize("dtype", [BF, F16])
def test_attention_and_norm(layout, dtype):
    from kohakuwullm_amd.kernels.elementwise.rmsnorm import rms_norm
    from kohakuwullm_amd.models.mlp import AttentionProjections
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    torch.manual_seed(SEED)
    block = AttentionProjections(256, 2, 1, 128).to(DEV).to(dtype)
    swap_mxfp8(block)
    x0, weight = _layouts(70, 256, dtype)[layout], torch.ones(256, device=DEV, dtype=dtype).requires_grad_()

    def run(train=True):
        x = x0.detach().requires_grad_(train)
        weight.grad = None
        block.zero_grad()
        with torch.set_grad_enabled(train):
            outs = [*block.project(rms_norm(x, weight))]
            outs.append(block.merge(outs[0]))
        if not train:
            return outs
        torch.autograd.backward(outs, [torch.ones_like(o).mul_(1e-2) for o in outs])
        return [o.detach() for o in outs] + [x.grad, weight.grad] + [p.grad for p in block.parameters()]

    _both(run)
    _both(lambda: run(False))


@pytest.mark.gpu
@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("dtype,autocast", [(BF, False), (F32, True)])
@pytest.mark.parametrize("tokens,hidden", [(1, 128), (97, 384), (64, 160)])
def test_feed_forward(fused, dtype, autocast, tokens, hidden):
    from kohakuwullm_amd.models.mlp import MXFP8SwiGLU, SwiGLU
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    if hidden % 128 and not fused:
        pytest.skip("a projection of this width is not swapped")
    torch.manual_seed(SEED)
    block = (MXFP8SwiGLU if fused else SwiGLU)(256, hidden=hidden).to(DEV).to(dtype)
    if not fused:
        swap_mxfp8(block)
    x0 = torch.randn(tokens, 256, device=DEV).to(dtype)

    def run(train=True):
        x = x0.detach().requires_grad_(train)
        block.zero_grad()
        with torch.autocast("cuda", dtype=BF, enabled=autocast), torch.set_grad_enabled(train):
            y = block(x)
        if not train:
            return [y]
        y.backward(torch.ones_like(y).mul_(1e-2))
        return [y.detach(), x.grad] + [p.grad for p in block.parameters()]

    _both(run)
    _both(lambda: run(False))


@pytest.mark.gpu
@pytest.mark.parametrize("tokens,shared,dtype", [(3, 0, BF), (130, 1, BF), (64, 0, F16)])
def test_mixture_of_experts(tokens, shared, dtype):
    from kohakuwullm_amd.models.moe import MoEMLP
    from kohakuwullm_amd.models.mxfp8_swap import swap_mxfp8

    torch.manual_seed(SEED)
    block = MoEMLP(256, hidden=128, num_experts=8, top_k=2, num_shared=shared).to(DEV).to(dtype)
    swap_mxfp8(block)
    x0 = torch.randn(tokens, 256, device=DEV).to(dtype)

    def run(train=True):
        x = x0.detach().requires_grad_(train)
        block.zero_grad()
        with torch.set_grad_enabled(train):
            y = block(x)
        if not train:
            return [y]
        y.backward(torch.ones_like(y).mul_(1e-2))
        # the gate's gradient is added with atomics in any order: what it reaches is compared below
        return [y.detach(), block.w_in.grad, block.w_out.grad], x.grad, block.router.weight.grad

    got, dx, dr = run()
    with _python():
        want, dx2, dr2 = run()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for a, b in ((dx, dx2), (dr, dr2)):  # fp32 sums of four terms in another order, rounded to 16 bits behind
        assert (a.float() - b.float()).norm() <= 4e-3 * b.float().norm()
    _both(lambda: run(False))


@pytest.mark.gpu
def test_refresh_and_pitched_products():
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, quantize_mx
    from kohakuwullm_amd.kernels.mxfp8.quantize import quantize_mx_dual_batch

    g = torch.Generator(device=DEV).manual_seed(SEED)
    ws = [torch.randn(m, k, device=DEV, generator=g).to(BF) for m, k in ((32, 32), (96, 256), (384, 128))] * 9  # two launches
    _both(lambda: [t for four in quantize_mx_dual_batch(ws) for t in four])
    q, s = quantize_mx(ws[1])
    _both(lambda: [mxfp8_matmul_pq(q, s, q, s, F32, out_pad=24)])


@pytest.mark.gpu
def test_threads_on_their_own_streams():
    """A launch and an allocation let other Python threads run: passes that overlap in time give what each gives alone."""
    import threading

    from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear

    torch.manual_seed(SEED)
    layers = [MXFP8Linear(512, 384 + 128 * i).to(DEV).to(BF) for i in range(4)]
    inputs = [torch.randn(300 + i, 512, device=DEV).to(BF) for i in range(4)]

    def run(lin, x0):
        x = x0.clone().requires_grad_()
        y = lin(x)
        dx, dw = torch.autograd.grad(y, [x, lin.weight], torch.full_like(y, 1e-2))
        return [y.detach(), dx, dw]

    want = [run(lin, x) for lin, x in zip(layers, inputs)]
    torch.cuda.synchronize()
    got = [[] for _ in layers]

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got[i].append(run(layers[i], inputs[i]))
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, passes in enumerate(got):
        assert len(passes) == 20
        for one in passes:
            assert all(torch.equal(_bits(a), _bits(b)) for a, b in zip(one, want[i]))


@pytest.mark.gpu
@pytest.mark.parametrize("way", ["extension", "ctypes"])
def test_threads_on_one_stream_share_the_scratch_of_k_splits(way):
    """Products whose partial sums go through the stream's one scratch tensor, issued by several threads at once: what each gives
    alone, bit for bit.  Ring slices, the dealt last round of large tiles, slices in a batch and the expert weight gradient."""
    import threading

    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, mxfp8_matmul_pq_batch
    from kohakuwullm_amd.kernels.mxfp8.grouped import grouped_mxfp8_wgrad, quantize_mx_cols_grouped

    g = torch.Generator(device=DEV).manual_seed(SEED)

    def operands(rows, k):
        codes = torch.randint(0, 120, (rows, k), device=DEV, generator=g, dtype=torch.uint8).view(torch.float8_e4m3fn)
        return codes, torch.randint(118, 126, (rows, k // 32), device=DEV, generator=g, dtype=torch.uint8)

    ring, dealt = ((*operands(m, k), *operands(n, k)) for m, n, k in ((300, 500, 8192), (1500, 4096, 16384)))
    both = [(*operands(3300, 8192), *operands(2500, 8192)), (*operands(2490, 8192), *operands(3310, 8192))]
    offsets = torch.tensor([0, 4000, 4000, 9000], dtype=torch.int32, device=DEV)
    rows = torch.randn(9000, 256, device=DEV, generator=g).to(BF)
    rq, rs = quantize_mx_cols_grouped(rows, offsets, 9000)
    jobs = [lambda: [mxfp8_matmul_pq(*ring, F32)], lambda: [mxfp8_matmul_pq(*dealt, BF)], lambda: mxfp8_matmul_pq_batch(both, BF),
            lambda: [grouped_mxfp8_wgrad(rq, rs, rq, rs, offsets, 9000)]]
    with contextlib.nullcontext() if way == "extension" else _python():
        want = [job() for job in jobs]
        torch.cuda.synchronize()
        got, start = [[] for _ in jobs], threading.Barrier(len(jobs))

        def work(i):
            start.wait()
            for _ in range(25):
                got[i].append(jobs[i]())

        threads = [threading.Thread(target=work, args=(i,)) for i in range(len(jobs))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        torch.cuda.synchronize()
    for i, passes in enumerate(got):
        assert len(passes) == 25
        for outs in passes:
            assert all(torch.equal(a, b) for a, b in zip(outs, want[i])), i


@pytest.mark.gpu
def test_scratch_belongs_to_the_binding():
    """Emptying its cache gives the memory back; the next product gets a scratch tensor anew, the same one from then on."""
    from kohakuwullm_amd import _lib
    from kohakuwullm_amd.kernels.mxfp8 import mxfp8_matmul_pq, quantize_mx

    q, s = quantize_mx(torch.randn(256, 8192, device=DEV).to(BF))
    want = mxfp8_matmul_pq(q, s, q, s, F32)
    size = int(_lib.load().mx_gemm_workspace_bytes())
    held = torch.cuda.memory_allocated()
    _lib._WORKSPACES.clear()
    assert held - torch.cuda.memory_allocated() >= size
    for _ in range(2):
        assert torch.equal(mxfp8_matmul_pq(q, s, q, s, F32), want)
        assert [t.numel() for t in _lib._WORKSPACES.values()] == [size]
