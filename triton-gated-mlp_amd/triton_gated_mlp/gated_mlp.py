"""Gated-MLP modules with the public surface of matteobonotto/triton-gated-mlp.

  FusedGatedMLP(hidden_size, intermediate_size, bias, hidden_act, dropout_p)   nn.Module, HIP kernels
  EagerGatedMLP(...)                                                           same math in plain torch
  FusedGatedMLPFunction.apply(x, W_up, b_up, W_gp, b_gp)                       hidden-state autograd op
  mlp_hidden_states_fwd / mlp_hidden_states_bwd, eager_fwd / eager_bwd, ACT_FWD

Reference: src/triton_gated_mlp/gated_mlp.py (EagerGatedMLP :73-98, eager_fwd/bwd :105-156,
FusedGatedMLPFunction :159-200, FusedGatedMLP :203-237).  Differences, all towards the eager
semantics: the fused path applies the gate/up/down biases and dropout (the reference drops them),
returns bias gradients, keeps G and U from the forward pass instead of recomputing them, runs the
down projection and its backward in the same kernels family (one autograd node for the MLP), and
implements every hidden_act of ACT_FWD (the reference's fused kernels know silu and no_act only).
"""

from __future__ import annotations

from typing import Optional

import torch
from torch import Tensor, nn
from torch.autograd.function import Function

from . import _cabi
from .ops import fwd as _fwd
from .ops.bwd import mlp_hidden_states_bwd
from .ops.fwd import mlp_hidden_states_fwd

class _FreshModule(dict):
    """Mapping name -> module class whose lookup hands out a NEW module instance (a value may be a
    (class, kwargs) pair): the behaviour of the reference's ACT2FN table
    (src/triton_gated_mlp/gated_mlp.py:10-26)."""

    def __getitem__(self, key):
        entry = super().__getitem__(key)
        cls, kwargs = entry if isinstance(entry, tuple) else (entry, {})
        return cls(**kwargs)


ACT2CLS = {name: type(mod) for name, mod in (
    ("gelu", nn.GELU()), ("leaky_relu", nn.LeakyReLU()), ("relu", nn.ReLU()), ("sigmoid", nn.Sigmoid()),
    ("silu", nn.SiLU()), ("swish", nn.SiLU()), ("tanh", nn.Tanh()))}
ACT2FN = _FreshModule(ACT2CLS)
ClassInstantier = _FreshModule  # the reference's name for it

ACT_FWD = {
    "gelu": nn.GELU(),
    "leaky_relu": nn.LeakyReLU(),
    "relu": nn.ReLU(),
    "sigmoid": nn.Sigmoid(),
    "silu": nn.SiLU(),
    "swish": nn.SiLU(),
    "tanh": nn.Tanh(),
    "no_act": nn.Identity(),
}


def _silu_op_bwd(x: Tensor, grad_output: Tensor) -> Tensor:
    sigma = torch.sigmoid(x)
    return grad_output * (sigma * (1 + x * (1 - sigma)))


ACT_BWD = {"silu": _silu_op_bwd, "swish": _silu_op_bwd}


class _GatedMLPBase(nn.Module):
    """Parameters and attributes shared by the eager and the fused module (same names, same order)."""

    def __init__(
        self,
        hidden_size: int = 256,
        intermediate_size: int = 512,
        bias: bool = True,
        hidden_act: str = "silu",
        dropout_p: float = 0.0,
    ):
        super().__init__()
        self.hidden_size = hidden_size
        self.intermediate_size = intermediate_size
        self.gate_proj = nn.Linear(hidden_size, intermediate_size, bias=bias)
        self.up_proj = nn.Linear(hidden_size, intermediate_size, bias=bias)
        self.down_proj = nn.Linear(intermediate_size, hidden_size, bias=bias)
        self.act = ACT_FWD[hidden_act]
        self.act_fn = hidden_act
        self.dropout = nn.Dropout(dropout_p)


class EagerGatedMLP(_GatedMLPBase):
    """down_proj(dropout(act(gate_proj(x)) * up_proj(x))) with stock torch operators."""

    def forward(self, x: Tensor) -> Tensor:
        lead = x.shape[:-1]
        x2 = x.reshape(-1, x.shape[-1])
        hidden = self.dropout(self.act(self.gate_proj(x2)) * self.up_proj(x2))
        return self.down_proj(hidden).reshape(*lead, self.hidden_size)


def eager_fwd(x: Tensor, WT_up: Tensor, b_up: Optional[Tensor], WT_gp: Tensor, b_gp: Optional[Tensor]) -> Tensor:
    """silu(x·W_gpᵀ + b_gp) * (x·W_upᵀ + b_up) in plain torch."""
    up = torch.nn.functional.linear(x, WT_up, b_up)
    gate = torch.nn.functional.linear(x, WT_gp, b_gp)
    return torch.nn.functional.silu(gate) * up


def eager_bwd(x: Tensor, W_up: Tensor, W_gp: Tensor, grad_output: Tensor):
    """Closed-form gradients (dx, dW_up, dW_gp) of eager_fwd without biases."""
    up = x @ W_up.T
    gate = x @ W_gp.T
    d_up = grad_output * torch.nn.functional.silu(gate)
    d_gate = _silu_op_bwd(gate, grad_output * up)
    return d_up @ W_up + d_gate @ W_gp, d_up.T @ x, d_gate.T @ x


_U64 = (1 << 64) - 1


class FusedGatedMLPFunction(Function):
    """Hidden-state operator hidden = dropout(act_fn(x·W_gpᵀ+b_gp) * (x·W_upᵀ+b_up)).

    Argument order (x, W_up, b_up, W_gp, b_gp) as in the reference; dropout_p, seed, offset and
    act_fn (default "silu") are optional.  `apply` records a native autograd node
    (csrc/torch_binding.cpp) that keeps G and U.
    """

    @staticmethod
    def apply(
        x: Tensor, W_up: Tensor, b_up: Optional[Tensor], W_gp: Tensor, b_gp: Optional[Tensor], dropout_p: float = 0.0,
        seed: int = 0, offset: int = 0, act_fn: str = "silu",
    ) -> Tensor:
        return _cabi.torch_binding().hidden(
            x, W_up, b_up, W_gp, b_gp, float(dropout_p), int(seed) & _U64, int(offset) & _U64, _cabi.act_code(act_fn)
        )


class FusedGatedMLPFullFunction(Function):
    """Whole MLP as one autograd node (native, csrc/torch_binding.cpp), so dY -> (dG, dU) is a single
    GEMM with a fused epilogue.  With `recompute` the node keeps only the inputs (as the reference does,
    gated_mlp.py:182) and runs the gate/up GEMM again in backward; the dropout mask is a function of
    the seed."""

    @staticmethod
    def apply(
        x: Tensor, W_gate: Tensor, b_gate: Optional[Tensor], W_up: Tensor, b_up: Optional[Tensor], W_down: Tensor,
        b_down: Optional[Tensor], dropout_p: float, seed: int, offset: int, recompute: bool = False, act_fn: str = "silu",
    ) -> Tensor:
        return _cabi.torch_binding().mlp_train(
            x, W_gate, b_gate, W_up, b_up, W_down, b_down, float(dropout_p), int(seed) & _U64, int(offset) & _U64,
            bool(recompute), _cabi.act_code(act_fn),
        )


class FusedGatedMLP(_GatedMLPBase):
    """Drop-in gated MLP running on hand-written gfx950 kernels (float16, bfloat16, or float32 with each
    operand split into three bf16 parts).  `hidden_act` is any key of ACT_FWD.

    Dropout is active in training mode only.  The keep mask comes from a counter-based generator:
    set `dropout_seed` (int) for a fixed mask stream, otherwise each forward draws a seed from
    torch's default CPU generator (so `torch.manual_seed` makes runs repeatable).  The seed and
    offset of the last training forward are kept in `last_dropout_state`; a batch that ran as
    several row chunks (see `_forward_rows`) drew one mask per chunk, and `last_dropout_states` lists
    them all as (first row, rows, seed, offset), the mask of a chunk being that of a [rows, N] tensor.

    Under `torch.autocast("cuda")` the module casts its input and parameters to the autocast dtype
    for the kernels (fp32 master weights keep fp32 gradients), as nn.Linear does.

    `recompute_activations = True` selects the memory-lean backward: only x is kept from the forward
    pass and G, U, H are recomputed (one more gate/up GEMM) instead of holding 3*M*N elements.
    """

    def __init__(self, *args, **kwargs):
        super().__init__(*args, **kwargs)
        self.dropout_seed: Optional[int] = None
        self.recompute_activations = False
        self._dropout_calls = 0
        self.last_dropout_state = (0, 0)
        self.last_dropout_states = []

    def _next_dropout_state(self):
        if self.dropout_seed is None:
            seed, offset = int(torch.randint(0, 2**62, (1,)).item()), 0
        else:
            seed, offset = int(self.dropout_seed), self._dropout_calls
            self._dropout_calls += 1
        self.last_dropout_state = (seed, offset)
        return seed, offset

    def forward(self, x: Tensor) -> Tensor:
        p = float(self.dropout.p) if self.training else 0.0
        self.last_dropout_states = []
        params = []
        for layer in (self.gate_proj, self.up_proj, self.down_proj):
            # (the usual parameters without a trip through nn.Module.__getattr__)
            own = layer._parameters
            params.append(own["weight"] if "weight" in own else layer.weight)
            params.append(own["bias"] if "bias" in own else layer.bias)
        if x.is_cuda and torch.is_autocast_enabled("cuda"):
            # Mixed precision as nn.Linear does it under torch.autocast: activations and (master)
            # weights are cast to the autocast dtype for the kernels; autograd casts the gradients back.
            with torch.autocast("cuda", enabled=False):
                dtype = torch.get_autocast_dtype("cuda")
                return self._forward_rows(x.to(dtype), [t if t is None else t.to(dtype) for t in params], p)
        return self._forward_rows(x, params, p)

    def _forward_rows(self, x: Tensor, params, p: float, row0: int = 0) -> Tensor:
        """x: [..., K]; params: weight and bias of gate, up and down."""
        K = x.shape[-1]
        M = x.numel() // K if K else 0
        limit = _fwd.max_rows_32bit(K, self.intermediate_size, x.dtype) if x.is_cuda else None
        if limit is not None and M > limit:
            # Token rows are independent: a batch too tall for the pipelined kernels' 32-bit operand
            # offsets runs as near-equal row chunks (autograd sums the chunks' weight gradients; with
            # dropout every chunk draws its own mask, recorded in `last_dropout_states`).
            chunks = -(-M // limit)
            rows = -(-M // (chunks * 256)) * 256
            x2 = x.reshape(-1, K)
            return torch.cat(
                [self._forward_rows(x2[i : i + rows], params, p, row0 + i) for i in range(0, M, rows)]
            ).reshape(x.shape)
        W_gate, b_gate, W_up, b_up, W_down, b_down = params
        graph = torch.is_grad_enabled() and (x.requires_grad or any(t is not None and t.requires_grad for t in params))
        if not graph and p == 0.0 and not torch._C._is_tracing():
            # Nothing to differentiate: the weight-streaming kernels for skinny M, no autograd node.  (A trace
            # records the operator below either way, which makes this choice whenever it runs.)
            return _cabi.torch_binding().mlp_infer(
                x, W_gate, b_gate, W_up, b_up, W_down, b_down, _cabi.act_code(self.act_fn)
            )
        if x.is_cuda and torch.cuda.is_current_stream_capturing():
            # Capturing forward + backward with torch.cuda.graph has ended in a host-side crash inside
            # the runtime's end-of-capture call on ROCm 7.2; until its cause is known the module
            # refuses rather than take the process down.  Inference forwards capture fine.
            raise RuntimeError(
                "FusedGatedMLP: capturing a step that records an autograd graph (training forward) into a "
                "HIP graph is not supported; capture inference forwards (torch.no_grad(), eval mode) only"
            )
        seed, offset = self._next_dropout_state() if p > 0.0 else (0, 0)
        if p > 0.0:
            self.last_dropout_states.append((row0, M, seed, offset))
        return FusedGatedMLPFullFunction.apply(
            x, W_gate, b_gate, W_up, b_up, W_down, b_down, p, seed, offset, self.recompute_activations, self.act_fn
        )
