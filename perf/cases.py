"""The work that users of this package have it do, as cases that can be timed.

A case is one pass through the public entry points: a training step of `FusedGatedMLP` (forward and
backward, every gradient), its inference forward (prompt processing and decoding), or a training step
of the hidden-state operator `FusedGatedMLPFunction`.

    M tokens, K hidden size, N intermediate size, any M >= 1, K and N multiples of 8

Inputs have the distributions that the benchmark and the tests state: x ~ N(0, 1), weights ~
N(0, 0.02), biases ~ U(-0.01, 0.01), upstream gradient ~ N(0, 1).  The package is imported from the
working folder, which is the root of the tree that is measured.
"""

from __future__ import annotations

import math
import os
import sys

import torch

_PACKAGE_DIR = os.path.join(os.getcwd(), "triton-gated-mlp_amd")
if _PACKAGE_DIR not in sys.path:
    sys.path.insert(0, _PACKAGE_DIR)

from triton_gated_mlp.gated_mlp import FusedGatedMLP, FusedGatedMLPFunction  # noqa: E402

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_SIZES = {"fp16": 2, "bf16": 2, "fp32": 4}


def _case(kind, dtype, M, K, N, bias=False, p=0.0, act="silu", recompute=False):
    return {"kind": kind, "dtype": dtype, "M": M, "K": K, "N": N, "bias": bias, "p": p, "act": act,
            "recompute": recompute}


def listed():
    named = [
        # the two ends of the reference benchmark's cube sweep that latency decides: launches and host
        # work at 32, a few kernels of a few microseconds at 512
        ("train_cube_32", _case("train", "fp16", 32, 32, 32)),
        ("train_cube_512", _case("train", "fp16", 512, 512, 512)),
        # an ordinary training step with every option a training configuration switches on
        ("train_mid_bias_dropout", _case("train", "bf16", 2048, 2048, 5632, bias=True, p=0.1)),
        # the headline training step, the largest case (Llama-3-8B widths)
        ("train_headline", _case("train", "fp16", 8192, 4096, 14336)),
        # odd token count, widths that no tile divides, biases, another activation
        ("train_ragged_gelu", _case("train", "bf16", 1357, 1160, 3096, bias=True, act="gelu")),
        # a model kept in float32, as the reference's own tests keep it
        ("train_fp32", _case("train", "fp32", 2048, 1024, 2816)),
        # the reference's autograd operator used on its own, the down projection left to the caller
        ("hidden_operator", _case("hidden", "fp16", 1024, 2048, 5632)),
        # a batch of prompts (Llama-2-7B widths) and one short prompt (Llama-3-8B widths)
        ("prefill_4096", _case("infer", "fp16", 4096, 4096, 11008)),
        ("prefill_short", _case("infer", "bf16", 200, 4096, 14336)),
        # decoding: a batch at Llama-3-70B widths, more sequences than one MFMA tile holds at 7B
        # widths, one sequence through a small model
        ("decode_batch_16", _case("infer", "fp16", 16, 8192, 28672)),
        ("decode_batch_24", _case("infer", "fp16", 24, 4096, 11008)),
        ("decode_single", _case("infer", "bf16", 1, 2048, 5632)),
    ]
    return [dict(case, name=name) for name, case in named]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _width(rng, lo, hi):
    """A layer width: as often a multiple of 256 (the usual kind) as any multiple of 8."""
    step = 256 if rng.random() < 0.5 and hi >= 512 else 8
    return max(step, round(_log_uniform(rng, lo, hi) / step) * step)


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["train", "train", "train", "infer", "infer", "hidden"])
    if kind == "infer":
        # from one token of one sequence to a batch of prompts
        dtype = rng.choice(["fp16", "bf16"])
        M = round(_log_uniform(rng, 1, 4096))
        K, most = _width(rng, 256, 8192), 6.0e12 / 3
    else:
        # from the sweep's smallest cube to the headline step
        dtype = rng.choice(["fp16", "fp16", "bf16", "bf16", "fp32"])
        M = round(_log_uniform(rng, 32, 8192))
        K = _width(rng, 32, 4096)
        most = 18.0 * 8192 * 4096 * 14336 / (12 if dtype == "fp32" else 1) / 1.5
    N = _width(rng, K, 4 * K)
    flops = (6.0 if kind == "infer" else 18.0) * M * K * N
    if flops > most:
        M = max(1, int(M * most / flops))
    bias = rng.random() < 0.4
    p = rng.choice([0.0, 0.0, 0.1]) if kind == "train" else 0.0
    act = rng.choice(["silu", "silu", "silu", "gelu", "relu"])
    recompute = kind == "train" and rng.random() < 0.15
    return _case(kind, dtype, M, K, N, bias=bias, p=p, act=act, recompute=recompute)


def prepare(case, seed):
    dtype = _DTYPES[case["dtype"]]
    M, K, N = case["M"], case["K"], case["N"]
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev).manual_seed(int(seed))

    def normal(shape, std, grad=False):
        t = torch.empty(shape, device=dev).normal_(0.0, std, generator=gen).to(dtype)
        return t.requires_grad_(grad)

    def uniform(shape, grad=False):
        t = torch.empty(shape, device=dev).uniform_(-0.01, 0.01, generator=gen).to(dtype)
        return t.requires_grad_(grad)

    training = case["kind"] != "infer"
    state = {"kind": case["kind"], "x": normal((M, K), 1.0, grad=training)}
    if case["kind"] == "hidden":
        state["W_up"], state["W_gate"] = normal((N, K), 0.02, grad=True), normal((N, K), 0.02, grad=True)
        state["b_up"] = uniform((N,), grad=True) if case["bias"] else None
        state["b_gate"] = uniform((N,), grad=True) if case["bias"] else None
        state["act"] = case["act"]
        state["dy"] = normal((M, N), 1.0)
        return state
    with torch.device(dev):
        mlp = FusedGatedMLP(hidden_size=K, intermediate_size=N, bias=case["bias"], hidden_act=case["act"],
                            dropout_p=case["p"]).to(dtype)
    with torch.no_grad():
        for layer in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
            layer.weight.copy_(normal(layer.weight.shape, 0.02))
            if layer.bias is not None:
                layer.bias.copy_(uniform(layer.bias.shape))
    if training:
        mlp.dropout_seed = int(seed)
        mlp.recompute_activations = case["recompute"]
        state["mlp"] = mlp.train()
        state["dy"] = normal((M, K), 1.0)
    else:
        state["mlp"] = mlp.eval()
    return state


def run(state):
    kind, x = state["kind"], state["x"]
    if kind == "infer":
        with torch.no_grad():
            return state["mlp"](x)
    if kind == "hidden":
        params = {n: state[n] for n in ("W_up", "b_up", "W_gate", "b_gate") if state[n] is not None}
        x.grad = None
        for t in params.values():
            t.grad = None
        extra = () if state["act"] == "silu" else (0.0, 0, 0, state["act"])
        y = FusedGatedMLPFunction.apply(x, state["W_up"], state["b_up"], state["W_gate"], state["b_gate"], *extra)
    else:
        mlp = state["mlp"]
        params = dict(mlp.named_parameters())
        x.grad = None
        mlp.zero_grad(set_to_none=True)
        y = mlp(x)
    y.backward(state["dy"])
    out = {name: t.grad for name, t in params.items()}
    out["x"] = x.grad
    out["y"] = y.detach()
    return out


def work(case):
    M, K, N, size = case["M"], case["K"], case["N"], _SIZES[case["dtype"]]
    weights = 2 * N * K + (2 * N if case["bias"] else 0)
    width = N
    if case["kind"] != "hidden":
        weights += K * N + (K if case["bias"] else 0)
        width = K
    if case["kind"] == "infer":
        # x and the weights in, y out
        return {"bytes": size * (M * K + weights + M * K), "flops": 6 * M * N * K}
    # x, dY and the weights in; y, dX and the weights' gradients out
    elements = 2 * M * K + 2 * M * width + 2 * weights
    return {"bytes": size * elements, "flops": (12 if case["kind"] == "hidden" else 18) * M * N * K}


def tolerance(case):
    # Four times what every output of the listed cases and of drawn ones differs by from the same
    # computation in float64 on the same rounded inputs (largest relative 2-norm seen over the outputs of
    # a pass: float32 1.6e-6, float16 3.9e-4, bfloat16 3.2e-3); for bfloat16 the 1e-2 that its 8 bits give.
    return {"rel": {"fp32": 1e-5, "fp16": 1.6e-3, "bf16": 1e-2}[case["dtype"]]}
