"""The work that users of this package have it do, as cases that can be prepared, run and compared.

A case is one pass of a module through its public entry points: an ``MXFP8Linear``, the GQA projections behind their
RMSNorm, the two forms of the SwiGLU feed-forward (the fused module, and the plain one after ``swap_mxfp8``), the
mixture-of-experts block after ``swap_mxfp8``, and the requantization of a model's weights between optimizer steps.
``train`` is forward and backward with every gradient, the other mode is a forward under ``no_grad``.  Widths are those
of the benchmark's configurations (and of the tests, for the small ones); token counts run from one sequence being
decoded to the benchmark's batches, whole blocks and ragged ones alike, because packed batches come in any length.
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from kohakuwullm_amd.kernels.elementwise.rmsnorm import rms_norm
from kohakuwullm_amd.kernels.mxfp8.linear import MXFP8Linear
from kohakuwullm_amd.models.mlp import AttentionProjections, MXFP8SwiGLU, SwiGLU
from kohakuwullm_amd.models.moe import MoEMLP
from kohakuwullm_amd.models.mxfp8_swap import refresh_mxfp8_weights, swap_mxfp8

DEVICE = "cuda"
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_HEAD_DIM = 128


def _linear(tokens, inp, out, train, dtype="bf16", autocast=False):
    return {"kind": "linear", "tokens": tokens, "inp": inp, "out": out, "train": train, "dtype": dtype, "autocast": autocast}


def _attention(tokens, dim, heads, kv_heads, train, dtype="bf16"):
    return {"kind": "attention", "tokens": tokens, "dim": dim, "heads": heads, "kv_heads": kv_heads, "train": train,
            "dtype": dtype, "autocast": False}


def _ffn(kind, tokens, dim, hidden, train, dtype="bf16", autocast=False):
    return {"kind": kind, "tokens": tokens, "dim": dim, "hidden": hidden, "train": train, "dtype": dtype, "autocast": autocast}


def _moe(tokens, dim, hidden, experts, top_k, shared, train, dtype="bf16"):
    return {"kind": "moe", "tokens": tokens, "dim": dim, "hidden": hidden, "experts": experts, "top_k": top_k,
            "shared": shared, "train": train, "dtype": dtype, "autocast": False}


def _refresh(blocks, dim, hidden, dtype="bf16"):
    return {"kind": "refresh", "blocks": blocks, "dim": dim, "hidden": hidden, "train": False, "dtype": dtype, "autocast": False}


def listed():
    return [
        # one decoding step of a small serving batch through one projection: latency, weights read once
        {"name": "linear_decode", **_linear(8, 2048, 3072, False)},
        # the small projection of the smoke configuration, trained: launches and host work weigh as much as the kernels
        {"name": "linear_train_small", **_linear(4096, 512, 1536, True)},
        # a packed fp16 batch of no round length, trained
        {"name": "linear_train_ragged", **_linear(3001, 2048, 2048, True, "fp16")},
        # the attention block's norm and four GQA projections at the benchmark's batch, trained: the largest case
        {"name": "attention_train", **_attention(32768, 2048, 16, 4, True)},
        # the same block decoding 64 sequences
        {"name": "attention_decode", **_attention(64, 2048, 16, 4, False)},
        # the dense feed-forward of the 546M-class model at the benchmark's batch, trained
        {"name": "ffn_train", **_ffn("ffn", 16384, 1536, 4096, True)},
        # the same block over one ragged prompt, forward only
        {"name": "ffn_prefill_ragged", **_ffn("ffn", 1500, 1536, 4096, False)},
        # an unmodified SwiGLU block after swap_mxfp8, fp32 masters and activations under bf16 autocast, ragged batch
        {"name": "swiglu_swapped_autocast_train", **_ffn("swiglu", 5003, 1536, 4096, True, "fp32", True)},
        # the 991M-class mixture of experts at the benchmark's batch (router, dispatch and routed experts), trained
        {"name": "moe_train", **_moe(16384, 1024, 512, 64, 6, 0, True)},
        # the same block with its shared expert (the constructor's default) on a small ragged batch, trained
        {"name": "moe_train_ragged", **_moe(2777, 1024, 512, 64, 6, 1, True)},
        # the same block decoding 32 sequences: few rows per expert, most experts' weights read
        {"name": "moe_decode", **_moe(32, 1024, 512, 64, 6, 1, False)},
        # both quantized copies of every linear weight of four blocks of the 546M-class model, once per optimizer step
        {"name": "weight_refresh", **_refresh(4, 1536, 4096)},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "attention", "ffn", "swiglu", "moe", "moe", "refresh"])
    train = rng.random() < 0.6
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    tokens = _log_int(rng, 128, 16384) if train else _log_int(rng, 1, 8192)
    if kind == "linear":
        inp, out = rng.choice([(512, 1536), (1536, 2560), (1536, 1536), (2048, 3072), (2048, 2048), (256, 1000), (2048, 512)])
        mixed = rng.random() < 0.3
        return _linear(tokens, inp, out, train, "fp32" if mixed else dtype, mixed)
    if kind == "attention":
        dim, heads, kv_heads = rng.choice([(2048, 16, 4), (1536, 12, 4), (512, 4, 2)])
        return _attention(tokens, dim, heads, kv_heads, train, dtype)
    if kind in ("ffn", "swiglu"):
        dim, hidden = rng.choice([(1536, 4096), (1536, 4096), (1024, 2816), (256, 512)])
        mixed = rng.random() < 0.4
        return _ffn(kind, tokens, dim, hidden, train, "fp32" if mixed else dtype, mixed)
    if kind == "moe":
        dim, hidden, experts, top_k = rng.choice([(1024, 512, 64, 6), (1024, 512, 64, 6), (1024, 512, 32, 8), (256, 128, 16, 4)])
        return _moe(tokens, dim, hidden, experts, top_k, rng.choice([0, 1]), train, dtype)
    return _refresh(rng.randint(1, 4), rng.choice([512, 1024, 1536]), rng.choice([2816, 3456, 4096]), dtype)


class _Attention(nn.Module):
    """The parts of an attention block around its core: norm weight and the four projections."""

    def __init__(self, dim, heads, kv_heads):
        super().__init__()
        self.norm = nn.Parameter(torch.ones(dim))
        self.proj = AttentionProjections(dim, heads, kv_heads, _HEAD_DIM)


def _build(case):
    kind = case["kind"]
    if kind == "linear":
        return MXFP8Linear(case["inp"], case["out"])
    if kind == "attention":
        return _Attention(case["dim"], case["heads"], case["kv_heads"])
    if kind == "ffn":
        return MXFP8SwiGLU(case["dim"], hidden=case["hidden"])
    if kind == "swiglu":
        return SwiGLU(case["dim"], hidden=case["hidden"])
    if kind == "moe":
        return MoEMLP(case["dim"], hidden=case["hidden"], num_experts=case["experts"], top_k=case["top_k"], num_shared=case["shared"])
    model = nn.ModuleList()
    for _ in range(case["blocks"]):
        model.append(MXFP8Linear(case["dim"], case["dim"] + 1024))
        model.append(MXFP8Linear(case["dim"], case["dim"]))
        model.append(MXFP8SwiGLU(case["dim"], hidden=case["hidden"]))
    return model


def prepare(case, seed):
    dtype = _DTYPES[case["dtype"]]
    act = torch.bfloat16 if case["autocast"] else dtype  # what leaves the block
    gen = torch.Generator(DEVICE).manual_seed(seed)

    def normal(*shape, std=1.0, to=dtype):
        return (torch.randn(*shape, generator=gen, device=DEVICE) * std).to(to)

    with torch.device(DEVICE):
        model = _build(case)
    model.to(dtype)
    with torch.no_grad():
        for p in model.parameters():
            if p.dim() == 1:
                p.copy_(1.0 + normal(*p.shape, std=0.1, to=torch.float32))
            else:
                p.copy_(normal(*p.shape, std=0.02, to=torch.float32))
        if case["kind"] == "moe":  # sharper scores than 0.02 gives: experts differ in load, as after some training
            model.router.weight.copy_(normal(*model.router.weight.shape, std=case["dim"] ** -0.5, to=torch.float32))
    if case["kind"] in ("attention", "swiglu", "moe"):
        swap_mxfp8(model)
    model.train(case["train"])
    refresh_mxfp8_weights(model)  # the quantized copies exist before the step, as after the last optimizer step
    state = {"case": case, "model": model, "params": list(model.parameters())}
    if case["kind"] == "refresh":
        return state
    tokens, train = case["tokens"], case["train"]
    state["x"] = normal(tokens, case["inp"] if case["kind"] == "linear" else case["dim"]).requires_grad_(train)
    if case["kind"] == "attention":
        shape = (case["heads"], _HEAD_DIM), (case["kv_heads"], _HEAD_DIM), (case["kv_heads"], _HEAD_DIM)
        state["heads"] = normal(tokens, case["heads"], _HEAD_DIM).requires_grad_(train)  # the attention core's output
        if train:
            state["upstream"] = [normal(tokens, *s, std=1e-2) for s in shape] + [normal(tokens, case["dim"], std=1e-2)]
    elif train:
        state["upstream"] = [normal(tokens, case["out"] if case["kind"] == "linear" else case["dim"], std=1e-2, to=act)]
    return state


def _forward(state):
    case, model, x = state["case"], state["model"], state["x"]
    if case["kind"] == "attention":
        return [*model.proj.project(rms_norm(x, model.norm)), model.proj.merge(state["heads"])]
    if case["autocast"]:
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return [model(x)]
    return [model(x)]


def run(state):
    case, model = state["case"], state["model"]
    if case["kind"] == "refresh":
        refresh_mxfp8_weights(model)
        copies = []
        for module in model:
            packed = module._packed if isinstance(module, MXFP8SwiGLU) else (module._cache,)
            copies += [t.view(torch.uint8) for pair in packed for t in pair]
        return copies
    if not case["train"]:
        with torch.no_grad():
            return _forward(state)
    leaves = [state["x"], *state["params"]] + ([state["heads"]] if "heads" in state else [])
    for leaf in leaves:
        leaf.grad = None
    load = [model.router.load_accum.zero_()] if case["kind"] == "moe" else []  # one step's rows per expert
    outputs = _forward(state)
    torch.autograd.backward(outputs, state["upstream"])
    return [t.detach() for t in outputs] + [leaf.grad for leaf in leaves] + load


def _live_experts(case):
    """Experts that get at least one row when the routing is near uniform."""
    rows = case["tokens"] * case["top_k"]
    return case["experts"] * (1.0 - (1.0 - 1.0 / case["experts"]) ** rows)


def work(case):
    kind = case["kind"]
    size = _DTYPES[case["dtype"]].itemsize
    code = 1.0 + 1.0 / 32.0  # bytes of one quantized element with its share of the block's scale
    if kind == "refresh":
        weights = case["blocks"] * (case["dim"] * (case["dim"] + 1024) + case["dim"] ** 2 + 3 * case["dim"] * case["hidden"])
        return {"bytes": weights * (size + 2 * code), "flops": 0.0}
    tokens, act = case["tokens"], 2 if case["autocast"] else size
    if kind == "linear":
        weights, macs, wide_in, wide_out = case["inp"] * case["out"], case["inp"] * case["out"], case["inp"], case["out"]
    elif kind == "attention":
        q, kv = case["heads"] * _HEAD_DIM, case["kv_heads"] * _HEAD_DIM
        weights = macs = case["dim"] * (2 * q + 2 * kv)
        wide_in, wide_out = case["dim"] + q, q + 2 * kv + case["dim"]
    elif kind in ("ffn", "swiglu"):
        weights = macs = 3 * case["dim"] * case["hidden"]
        wide_in = wide_out = case["dim"]
    else:
        one = 3 * case["dim"] * case["hidden"]
        router = case["dim"] * case["experts"]
        # weights: what a forward must read; every expert's gradient is written
        weights = one * (_live_experts(case) + case["shared"]) + router
        macs = one * (case["top_k"] + case["shared"]) + router
        wide_in = wide_out = case["dim"]
    if not case["train"]:
        return {"bytes": tokens * (wide_in * size + wide_out * act) + weights * code, "flops": 2.0 * tokens * macs}
    grads = weights if kind != "moe" else 3 * case["dim"] * case["hidden"] * (case["experts"] + case["shared"])
    return {"bytes": 2 * tokens * (wide_in * size + wide_out * act) + 2 * weights * code + grads * size, "flops": 6.0 * tokens * macs}


def tolerance(case):
    if case["kind"] == "refresh":
        return "exact"  # codes and scale bytes
    # Against fp64 on the same quantized operands one product is 1.7e-3 off, the rounding of its 16-bit output; the
    # backward stacks two of those, and sums of 16-bit partial results (dx of the three projections of one input, dW
    # rounded before it is widened to an fp32 master) may be rounded once or once per term: 2.4e-3 to 3e-3.  The order
    # of the sums alone changes 1e-4 at most (contraction axes permuted in blocks of 128, every listed case).
    return {"rel": 1e-2}
