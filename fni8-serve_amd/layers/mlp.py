"""Gated MLP over two W8A8 linears (fni8serve/layers/mlp.py:22-48).

`GatedMLP(gate_up, down, *, act="silu", bias_gate_up=None, bias_down=None)`
computes down(act_and_mul(gate_up(x))) with gate/up merged into one
[2*intermediate, hidden] weight (mlp.py:39-40).  On the GPU, with int8
weights, a kernel activation (silu, tanh gelu) and at least FUSE_MIN_ROWS
rows, the activation and the down projection's per-token quantization run as
one launch (`ops.act_and_mul_quant`) feeding the int8 GEMM directly: the fp16
[M, intermediate] tensor never goes to HBM, and the result is bit-identical to
the unfused chain.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules.module import _has_any_global_hook

from .. import ops
from ..qtensor import QTensor
from .activation import GeluAndMul, SiluAndMul, fused_act, get_act_and_mul
from .linear import LinearW8A8

# Rows from which the fused activation + quantization feeds the down projection.
# Below it the unfused chain is faster: up to 4 rows the down projection's
# linear() quantizes its own input inside the GEMM at almost no cost, while the
# fused kernel runs each row's activation (12288 exps for Qwen3-8B) on one
# workgroup (MI355X, Qwen3-8B down chain, unfused vs fused: 10.07 vs 11.66 us at
# 1 row, 12.54 vs 14.69 at 4; 15.81 vs 15.50 at 16, 26.73 vs 26.09 at 64).
FUSE_MIN_ROWS = 5


# What calling one of these modules runs, as their classes were defined: forward and, in
# a linear, the rule that it asks.
_CALL = getattr(nn.Module, "_wrapped_call_impl", None)
_DEFINED = {cls: (cls.forward, getattr(cls, "_int8_ok", None))
            for cls in (LinearW8A8, SiluAndMul, GeluAndMul)}


def bare(m: nn.Module, cls: type) -> bool:
    """True when calling `m` is calling the forward that `cls` was defined with and nothing
    else, but for hooks on every module: exactly that class, no hook on it, not compiled,
    and no method of its own or put on the class since."""
    d = m.__dict__
    forward, rule = _DEFINED.get(cls, (None, None))
    return (type(m) is cls and cls.forward is forward and cls.__call__ is _CALL
            and "forward" not in d and "_compiled_call_impl" not in d
            and (rule is None or (cls._int8_ok is rule and "_int8_ok" not in d))
            and not (d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"]
                     or d["_backward_pre_hooks"]))


class GatedMLP(nn.Module):
    def __init__(self, gate_up: QTensor, down: QTensor, *, act: nn.Module | str = "silu",
                 bias_gate_up=None, bias_down=None):
        super().__init__()
        self.gate_up_proj = LinearW8A8(gate_up, bias_gate_up)
        self.down_proj = LinearW8A8(down, bias_down)
        self.act_fn = get_act_and_mul(act) if isinstance(act, str) else act
        self.hidden_size = self.down_proj.out_features
        self.intermediate_size = self.gate_up_proj.out_features // 2

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        gate_up, down, act_fn = self.gate_up_proj, self.down_proj, self.act_fn
        act = fused_act(act_fn)
        if (act is not None and x.is_cuda and not _has_any_global_hook()
                and bare(gate_up, LinearW8A8) and bare(down, LinearW8A8)
                and bare(act_fn, type(act_fn))):
            y = ops.gated_mlp(x, gate_up.weight, down.weight, act, gate_up.bias, down.bias,
                              FUSE_MIN_ROWS)
            if y is not None:
                return y
        rows = x.numel() // max(x.shape[-1], 1)
        if act is not None and rows >= FUSE_MIN_ROWS and gate_up._int8_ok(x) and down._int8_ok(x):
            h = gate_up(x)
            xq, xs = ops.act_and_mul_quant(h, act)
            y = ops.gemm_quantized(xq, xs, down.weight, down.bias)
            return y.reshape(*x.shape[:-1], y.shape[-1])
        return down(act_fn(gate_up(x)))


class Qwen3MLP(GatedMLP):
    """Qwen3 dense MLP (SwiGLU)."""

    def __init__(self, gate_up: QTensor, down: QTensor, bias_gate_up=None, bias_down=None):
        super().__init__(gate_up, down, act=SiluAndMul(), bias_gate_up=bias_gate_up,
                         bias_down=bias_down)
