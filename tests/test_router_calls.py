"""Which calls the router's kernels may stand for, decided on the host: what does not fit goes to the PyTorch composition."""

import pytest
import torch

from conftest import SEED

BF, HF, F32 = torch.bfloat16, torch.float16, torch.float32


def _operands(tokens=4, dim=64, experts=16, xdt=BF, wdt=BF):
    return torch.zeros(tokens, dim, dtype=xdt), torch.zeros(experts, dim, dtype=wdt)


def test_operands_that_fit():
    from kohakuwullm_amd.kernels.moe.router import can_route, operands_fit

    for xdt, wdt in ((BF, BF), (HF, HF), (F32, F32), (BF, F32), (HF, F32)):
        x, w = _operands(xdt=xdt, wdt=wdt)
        assert operands_fit(x, w, 4)
        assert not can_route(x, w, 4)  # on the CPU


@pytest.mark.parametrize("width", [8, 56, 72, 128])
def test_input_of_another_width_is_refused(width):
    """The kernels index the router matrix by the input's width: a wider input read past the matrix, and the backward wrote
    past its gradient."""
    from kohakuwullm_amd.kernels.moe.router import operands_fit, route_topk

    x, w = torch.zeros(4, width, dtype=BF), _operands()[1]
    assert not operands_fit(x, w, 4)
    with pytest.raises(ValueError):
        route_topk(x, w, None, 4, True, 1.0)


def test_other_operands_are_refused():
    from kohakuwullm_amd.kernels.moe.router import operands_fit

    x, w = _operands()
    assert not operands_fit(x[0], w, 4) and not operands_fit(x[:0], w, 4) and not operands_fit(x, w.view(16, 8, 8), 4)
    assert not operands_fit(x, w, 0) and not operands_fit(x, w, 17)
    assert not operands_fit(x.double(), w, 4) and not operands_fit(x.float(), w, 4) and not operands_fit(x, w.half(), 4)
    assert not operands_fit(*_operands(dim=60), 4) and not operands_fit(*_operands(experts=257), 4)
    assert not operands_fit(x, torch.zeros(64, 16, dtype=BF).t(), 4)
    assert not operands_fit(x, torch.zeros(16 * 64 + 1, dtype=BF)[1:].view(16, 64), 4)


def test_operands_past_the_grid_are_refused():
    """Token counts and widths that the backward, or either direction, has no launch for; the composition takes them."""
    from kohakuwullm_amd.kernels.moe.router import operands_fit

    def fits(tokens, dim):
        return operands_fit(torch.empty(tokens, dim, dtype=BF, device="meta"), torch.empty(8, dim, dtype=BF, device="meta"), 2)

    assert fits(65535 * 256, 64) and not fits(65535 * 256 + 1, 64)
    assert fits(4, (1 << 24) - 8) and not fits(4, 1 << 24)


def test_bias_that_is_not_the_kernels_is_refused():
    """The selection bias reaches the kernels as a pointer: its length, type, layout and device are checked on the host."""
    from kohakuwullm_amd.kernels.moe.router import operands_fit, route_topk

    x, w = _operands()
    for dtype in (BF, HF, F32):
        assert operands_fit(x, w, 4, torch.zeros(16, dtype=dtype))
    for bias in (torch.zeros(16, dtype=torch.float64), torch.zeros(15), torch.zeros(1, 16), torch.zeros(1), torch.zeros(32)[::2],
                 torch.zeros(1).expand(16), torch.zeros(16, device="meta")):
        assert not operands_fit(x, w, 4, bias)
        with pytest.raises(ValueError):
            route_topk(x, w, bias, 4, True, 1.0)


def test_traced_and_transformed_calls_are_composed():
    """Calls that someone traces, maps or differentiates forward are left to operators those can see."""
    from torch.autograd import forward_ad
    from torch.utils._python_dispatch import TorchDispatchMode

    from kohakuwullm_amd.kernels.moe.router import plain_call

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    x, seen = torch.zeros(2, 3), []
    note = lambda t: (seen.append(plain_call(t)), t * 1.0)[1]  # noqa: E731
    assert plain_call(x, torch.nn.Parameter(x))
    torch.func.vmap(note)(x)
    torch.func.jvp(note, (x,), (x,))
    torch.func.grad(lambda t: note(t).sum())(x)
    torch.jit.trace(note, x, check_trace=False)
    with forward_ad.dual_level():
        note(forward_ad.make_dual(x, x))
    with Seen():
        note(x)
    assert seen == [False] * 6
    assert not plain_call(x.as_subclass(Sub)) and plain_call(x)


@pytest.mark.parametrize("norm", [False, True])
def test_composed_gradients(norm):
    """The backward's operators against autograd's of the forward, once and twice differentiated."""
    from kohakuwullm_amd.kernels.moe.router import composed_gradients

    torch.manual_seed(SEED)
    x, w, up = (torch.randn(*s).requires_grad_(True) for s in ((5, 8), (6, 8), (5, 3)))
    scores = (x @ w.T).sigmoid()
    idx = scores.topk(3, dim=-1).indices
    gate = scores.gather(1, idx)
    gate = 1.5 * (gate / gate.sum(-1, keepdim=True).clamp_min(1e-9) if norm else gate)
    want = torch.autograd.grad(gate, [x, w], up, create_graph=True)
    got = composed_gradients(up, x, w, idx, norm, 1.5)
    # fp32 sums of at most 8 terms of size 1, a few roundings each: 64 units of 2^-24 bound both orders
    close = lambda a, b: torch.allclose(a, b, rtol=64 * 2.0**-24, atol=64 * 2.0**-24)  # noqa: E731
    assert all(close(a, b) for a, b in zip(got, want))
    twice = [torch.autograd.grad(sum(t.pow(2).sum() for t in ts), [x, w, up], retain_graph=True) for ts in (got, want)]
    assert all(torch.allclose(a, b, rtol=1e-4, atol=1e-5) for a, b in zip(*twice))  # a second derivative: ten such sums deep


@pytest.mark.parametrize("layout", ["offset", "strides"])
def test_backward_of_operands_that_a_hook_laid_out_anew(monkeypatch, layout):
    """Saved-tensor hooks may give the operands back at an odd offset or in another order of strides; the kernels get pointers."""
    import ctypes
    from types import SimpleNamespace

    from kohakuwullm_amd.kernels.moe import router

    seen = {}

    def invoke(name, work, like, *args):
        if name == "mx_router_topk_backward":
            for key, at, size in (("idx", 2, 5 * 3 * 8), ("scores", 3, 5 * 3 * 4), ("x", 4, 5 * 8 * 4), ("weight", 7, 6 * 8 * 4)):
                seen[key] = args[at] % 16, ctypes.string_at(args[at], size)

    monkeypatch.setattr(router, "_lib", SimpleNamespace(
        MX_DTYPE=router._lib.MX_DTYPE, invoke=invoke, load=lambda: SimpleNamespace(mx_router_backward_workspace=lambda *a: 1)))
    kept = []

    def pack(t):
        kept.append(t.detach())
        return t

    def unpack(t):
        t = t.detach()
        if layout == "strides":
            return t.t().contiguous().t()
        return t.new_empty(t.numel() + 1)[1:].view(t.shape).copy_(t)

    torch.manual_seed(SEED)
    x, w = torch.randn(5, 8).requires_grad_(True), torch.randn(6, 8).requires_grad_(True)
    with torch.autograd.graph.saved_tensors_hooks(pack, unpack):
        gate = router.route_topk(x, w, None, 3, True, 1.0)[1]
    kept[2].copy_(torch.arange(15).view(5, 3) % 6)  # nobody wrote them: no kernel ran
    kept[3].copy_(torch.arange(15.0).view(5, 3))
    gate.backward(torch.ones(5, 3))
    for key, t in zip(("x", "weight", "idx", "scores"), kept):
        assert seen[key][1] == t.contiguous().numpy().tobytes(), key
    assert seen["x"][0] == 0 and seen["weight"][0] == 0
