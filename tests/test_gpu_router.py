"""The fused top-k router against fp64 on the CPU: selection, gate weights, histogram and both gradients, at the edges of
its tiles (tokens per workgroup 16, 32 or 64 by their number, experts per MFMA tile 16 and per lane 64, K steps of 32 over eight waves, chunks of
tokens and 128 columns in the backward)."""

import pytest
import torch

from conftest import SEED

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("tokens,dim,experts,top_k,xdt,wdt,norm,biased", [
    (1, 8, 1, 1, BF, BF, False, False),
    (16, 256, 64, 6, BF, BF, True, True),
    (17, 72, 16, 4, BF, F32, True, True),
    (50, 1024, 33, 8, HF, HF, True, False),
    (300, 520, 100, 16, F32, F32, False, True),
    (130, 136, 256, 5, HF, F32, True, True),
    (5003, 1024, 64, 6, BF, BF, True, True),
    (12301, 136, 48, 4, HF, HF, True, True),
    (33001, 16, 17, 16, BF, BF, True, False),  # five tokens for a wave of the dx kernel, whole chunks of 256 tokens and 16 picks
])
def test_route_topk(tokens, dim, experts, top_k, xdt, wdt, norm, biased):
    from kohakuwullm_amd.kernels.moe.router import can_route, route_topk

    g = torch.Generator().manual_seed(SEED)
    x = torch.randn(tokens, dim, generator=g).to(xdt)
    w = (torch.randn(experts, dim, generator=g) * dim**-0.5).to(wdt)
    bias = (torch.randn(experts, generator=g) * 0.05).to(BF) if biased else None
    up = torch.randn(tokens, top_k, generator=g).to(xdt)
    xd, wd = x.to(DEV).requires_grad_(True), w.to(DEV).requires_grad_(True)
    assert can_route(xd, wd, top_k)
    idx, gate, counts = route_topk(xd, wd, None if bias is None else bias.to(DEV), top_k, norm, 1.5)
    assert idx.dtype == torch.int64 and gate.dtype == xdt and counts.dtype == torch.int32

    x64, w64 = x.double().requires_grad_(True), w.double().requires_grad_(True)
    scores = (x64 @ w64.T).sigmoid()
    choose = scores.detach() + (0.0 if bias is None else bias.double())
    want = choose.topk(top_k, dim=-1).indices
    got = idx.cpu()
    # a different pick is a near tie: an fp32 sum of `dim` products of size ~1/sqrt(dim) and the sigmoid are off by less
    # than 2^-24 (sqrt(dim) + 8) here, and the two picks' scores differ by no more than twice that
    bound = 2.0 ** -23 * (dim**0.5 + 8)
    gap = (choose.gather(1, got) - choose.gather(1, want)).abs()
    assert (gap[got != want] < bound).all()
    assert torch.equal(counts.cpu().long(), torch.bincount(got.reshape(-1), minlength=experts))
    picked = scores.gather(1, got)
    ref = 1.5 * (picked / picked.sum(-1, keepdim=True) if norm else picked)
    # half a unit in the last place, relative: 2^-p for a significand of p bits (8, 11, 24), plus the fp32 error of the logit
    half_ulp = {BF: 2.0**-8, HF: 2.0**-11, F32: 2.0**-24}
    assert ((gate.detach().cpu().double() - ref.detach()).abs() <= ref.detach() * half_ulp[xdt] * 1.01 + bound).all()

    gate.backward(up.to(DEV))
    ref.backward(up.double())
    for mine, theirs, dtype in ((xd.grad, x64.grad, xdt), (wd.grad, w64.grad, wdt)):
        assert mine.dtype == dtype
        err = (mine.cpu().double() - theirs).norm() / theirs.norm().clamp_min(1e-30)
        # rounding to the output type, and fp32 sums whose terms carry a few relative roundings each
        assert err <= half_ulp[dtype] + 2.0**-24 * (tokens**0.5 + 64), (err, dtype)


def test_router_module_on_kernels_matches_its_composition():
    """TopKRouter with the kernels and with its PyTorch composition (the same call under a group count it composes)."""
    from kohakuwullm_amd.models.moe import TopKRouter

    torch.manual_seed(SEED)
    router = TopKRouter(256, 32, top_k=4).to(DEV)
    router.expert_bias.normal_(std=0.02)
    x = torch.randn(700, 256, device=DEV)
    idx, gate, counts = router.route(x)
    router.z_loss_weight = 1e-6  # an auxiliary term: the composition
    ref_idx, ref_gate, ref_counts = router.route(x)
    router.z_loss_weight = 0.0
    assert torch.equal(idx, ref_idx) and torch.equal(counts, ref_counts)
    assert torch.allclose(gate, ref_gate, rtol=1e-5, atol=0)
    assert torch.equal(router.load_accum, 2.0 * counts)
    with torch.no_grad():
        assert torch.equal(router.route(x)[1], gate)


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("what", [float("nan"), float("inf"), -float("inf")])
def test_scores_that_are_not_finite(what, dtype):
    """One expert whose scores are NaN or saturated: picks, gates and gradients are not finite where the composition's are not."""
    from kohakuwullm_amd.models.moe import TopKRouter

    torch.manual_seed(SEED)
    router = TopKRouter(64, 16, top_k=4).to(DEV).to(dtype)
    x = torch.randn(40, 64, device=DEV).abs().to(dtype).requires_grad_(True)
    up = torch.randn(40, 4, device=DEV).to(dtype)
    with torch.no_grad():
        router.weight[5, 7] = what
    results = []
    for z_loss_weight in (0.0, 1e-6):  # kernels, composition
        router.z_loss_weight = z_loss_weight
        idx, gate, counts = router.route(x)
        results.append([idx, counts, gate.detach(), *torch.autograd.grad(gate, [x, router.weight], up)])
    for name, a, b in zip(("idx", "counts", "gate", "dx", "dw"), *results):
        if not a.is_floating_point():
            assert torch.equal(a, b)
            continue
        if name == "dx" and what == -float("inf"):
            # nobody picks that expert: its gradient of 0 is no term of the kernel's dx, in the dense product it is 0 * inf
            assert a.isfinite().all()
            a = torch.where(b.isnan(), b, a)
        assert torch.equal(a.isnan(), b.isnan()), name
        # rounding to the type (2^-8 at most), and fp32 sums of 64 products
        assert torch.allclose(a.float().nan_to_num(), b.float().nan_to_num(), rtol=2.0**-7, atol=2.0**-7), name


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("tokens", [1, 37])
def test_route_takes_any_layout(tokens, dtype):
    """Views at odd offsets, pitched and broadcast rows: the result and gradients of an aligned copy."""
    from kohakuwullm_amd.kernels.moe.router import route_topk

    torch.manual_seed(SEED)
    w = torch.randn(16, 64, device=DEV).to(dtype).requires_grad_(True)
    flat, wide = torch.randn(tokens * 64 + 1, device=DEV).to(dtype), torch.randn(tokens, 68, device=DEV).to(dtype)
    up = torch.randn(tokens, 4, device=DEV).to(dtype)

    def step(x):
        x = x.detach().requires_grad_(True)
        idx, gate, counts = route_topk(x, w, None, 4, True, 1.0)
        return [idx, gate.detach(), counts, *torch.autograd.grad(gate, [x, w], up)]

    for x in (flat[1:].view(tokens, 64), wide[:, :64], flat[:64].expand(tokens, 64), flat[: tokens * 64].view(64, tokens).t()):
        for a, b in zip(step(x), step(x.clone(memory_format=torch.contiguous_format))):
            assert torch.equal(a, b)


@pytest.mark.parametrize("norm", [False, True])
def test_route_differentiated_twice_batched_and_forward(norm):
    """create_graph, batched upstream gradients and forward mode give what the composition gives."""
    from torch.autograd import forward_ad

    from kohakuwullm_amd.models.moe import TopKRouter

    torch.manual_seed(SEED)
    router = TopKRouter(64, 16, top_k=4, norm_topk_prob=norm).to(DEV)
    x = torch.randn(20, 64, device=DEV).requires_grad_(True)
    up, ups = torch.randn(20, 4, device=DEV), torch.randn(3, 20, 4, device=DEV)
    leaves = [x, router.weight]

    def results():
        gate = router.route(x)[1]
        first = torch.autograd.grad(gate, leaves, up, create_graph=True)
        second = torch.autograd.grad(sum(t.pow(2).sum() for t in first), leaves, retain_graph=True)
        mapped = torch.autograd.grad(gate, leaves, ups, is_grads_batched=True)
        return [gate, *first, *second, *mapped]

    got, kernel_name = results(), type(router.route(x)[1].grad_fn).__name__
    with torch.no_grad(), forward_ad.dual_level():
        tangent = forward_ad.unpack_dual(router.route(forward_ad.make_dual(x.detach(), torch.ones_like(x)))[1]).tangent
    router.z_loss_weight = 1e-6  # an auxiliary term: the composition throughout
    want = results()
    assert kernel_name == "_RouteTopKBackward"
    # fp32 sums of 64 products of size 1 in another order, two derivatives deep
    for a, b in zip(got, want):
        assert torch.allclose(a, b, rtol=1e-4, atol=1e-5)
    with torch.no_grad(), forward_ad.dual_level():
        ref = forward_ad.unpack_dual(router.route(forward_ad.make_dual(x.detach(), torch.ones_like(x)))[1]).tangent
    assert torch.equal(tangent, ref)


def test_router_bias_of_another_type_is_composed():
    """An fp64 bias was accepted by the composition and is again (the kernels know 16-bit and fp32 ones)."""
    from kohakuwullm_amd.models.moe import TopKRouter

    torch.manual_seed(SEED)
    router = TopKRouter(128, 16, top_k=4).to(DEV)
    router.expert_bias.normal_(std=0.02)
    x = torch.randn(50, 128, device=DEV)
    idx, gate, counts = router.route(x)
    router.expert_bias = router.expert_bias.double()
    again = router.route(x)
    assert torch.equal(again[0], idx) and torch.equal(again[2], counts) and torch.allclose(again[1], gate, rtol=1e-5, atol=0)


def test_router_of_another_width_raises():
    """A block whose router reads another width than it is given: an error, as the composition's product raises it."""
    from kohakuwullm_amd.models.moe import MoEMLP

    block = MoEMLP(256, hidden=128, num_experts=16, top_k=4, num_shared=0, router_dim=128).to(DEV).to(BF)
    x = torch.randn(40, 256, device=DEV).to(BF)
    with pytest.raises(RuntimeError):
        block(x)
    with pytest.raises(RuntimeError):
        block(x, route_on=x[:, :64])
    assert block(x, route_on=x[:, :128].contiguous()).shape == x.shape


@pytest.mark.parametrize("dtype", [BF, HF, F32])
@pytest.mark.parametrize("tokens,dim,top_k", [(1, 8, 1), (37, 520, 3), (9000, 256, 6)])
@pytest.mark.parametrize("layout", ["plain", "pitched", "transposed", "broadcast", "none"])
def test_gradient_that_comes_through_the_router(tokens, dim, top_k, dtype, layout):
    """``through``: what x's further use gives is added to the router's gradient in its kernel, however it lies."""
    from kohakuwullm_amd.kernels.moe.router import route_fitting

    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.randn(tokens, dim, device=DEV, generator=g).to(dtype).requires_grad_()
    w = (torch.randn(16, dim, device=DEV, generator=g) * dim**-0.5).to(dtype).requires_grad_()
    up = torch.randn(tokens, top_k, device=DEV, generator=g).to(dtype)
    onto = torch.randn(tokens, dim, device=DEV, generator=g).to(dtype)
    onto = {"plain": onto, "pitched": torch.empty(tokens, dim + 4, device=DEV, dtype=dtype)[:, :dim].copy_(onto),
            "transposed": onto.t().contiguous().t(), "broadcast": onto[:1].expand(tokens, dim), "none": None}[layout]
    plain = torch.autograd.grad(route_fitting(x, w, None, top_k, True, 1.5)[1], [x, w], up)
    idx, gate, counts, same = route_fitting(x, w, None, top_k, True, 1.5, True)
    assert same.data_ptr() == x.data_ptr() and torch.equal(same, x)
    if onto is None:
        dx, dw = torch.autograd.grad(gate, [x, w], up)
        assert torch.equal(dx, plain[0]) and torch.equal(dw, plain[1])
        return
    dx, dw = torch.autograd.grad([gate, same], [x, w], [up, onto], retain_graph=True)
    assert torch.equal(dw, plain[1])
    # the gradient itself and the sum rounded once each on one side, the sum alone on the other
    unit = {BF: 2.0**-8, HF: 2.0**-11, F32: 2.0**-23}[dtype]
    want = plain[0].double() + onto.double()
    # ... and fp32 sums of top_k terms of up to 3 max|up| max|w| (s / S <= 1) and `onto`, in another order
    terms = top_k * 3.0 * up.abs().max().double() * w.detach().abs().max().double()
    assert ((dx.double() - want).abs() <= unit * (plain[0].double().abs() + want.abs()) + 2.0**-21 * (terms + onto.double().abs())).all()
    assert torch.equal(torch.autograd.grad(same, x, onto, retain_graph=True)[0], onto)  # the gate weights unused
    again = torch.autograd.grad([gate, same], [x, w], [up, onto], create_graph=True)  # by operators
    assert again[0].requires_grad and (again[0].double() - want).norm() <= 4 * unit * want.norm() + 1e-5 * want.norm()


@pytest.mark.parametrize("dim,top_k,xdt,wdt,norm", [(520, 16, BF, BF, True), (8, 1, HF, F32, False), (512, 9, F32, F32, True), (1032, 6, HF, HF, True)])
def test_dx_of_many_tokens(dim, top_k, xdt, wdt, norm):
    """Past the count from which sixteen tokens share a workgroup: bit for bit the dx that the same tokens get in short batches."""
    from kohakuwullm_amd.kernels.moe.router import route_fitting

    g = torch.Generator(device=DEV).manual_seed(SEED)
    tokens = (32 if dim <= 512 else 48) * torch.cuda.get_device_properties(DEV).multi_processor_count + 5
    x = torch.randn(tokens, dim, device=DEV, generator=g).to(xdt).requires_grad_()
    w = (torch.randn(48, dim, device=DEV, generator=g) * dim**-0.5).to(wdt).requires_grad_()
    up = torch.randn(tokens, top_k, device=DEV, generator=g).to(xdt)
    onto = torch.randn(tokens, dim + 8, device=DEV, generator=g).to(xdt)[:, :dim]

    def gradients(rows):
        part = x[rows]
        _, gate, _, same = route_fitting(part, w, None, top_k, norm, 1.5, True)
        alone = torch.autograd.grad(gate, part, up[rows], retain_graph=True)[0]
        return alone, torch.autograd.grad([gate, same], part, [up[rows], onto[rows]])[0]

    whole = gradients(slice(None))
    for lo in range(0, tokens, 5000):
        rows = slice(lo, min(lo + 5000, tokens))
        for a, b in zip(whole, gradients(rows)):
            assert torch.equal(a[rows], b)
