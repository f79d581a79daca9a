"""Fused channel-mix building blocks (HIP kernels) as autograd Functions.

RWKV6ChannelMix.forward (/root/reference/rwkv_megatron/rwkv6_layer_specs.py:512-536):

    delta = shift(x) - x                                   :513-516
    mixed_up, mixed_gate = x + delta * mix_coeffs[e]       :517-520
    h = relu(linear_up(mixed_up)) ** 2                     :522-524
    out = linear_down(h)                                   :525
    y = out * sigmoid(linear_gate(mixed_gate))             :528-536

* ``cmix_lerp``: the shift and both lerps in one pass, written as two separate [T,B,C]
  tensors, each a contiguous GEMM operand (the reference's ``unbind`` + ``.contiguous()``
  copies, and the stack of their gradients, disappear).  Its backward is one pass
  producing dx and d mix_coeffs from the two gradients where they lie.
* ``relu_sq`` and ``sigmoid_gate``: single-pass epilogues with single-pass backwards.

The projections stay on hipBLASLt (torch.nn.functional.linear).  Every function raises
if the HIP library is missing; there is no fallback.  The autograd functions are
csrc/autograd.cpp's.
"""
from __future__ import annotations

import torch

from . import _lib
from .timemix import _check_act

NE = 2  # (up, gate)


def cmix_lerp(x: torch.Tensor, mix: torch.Tensor) -> torch.Tensor:
    """[T,B,C] bf16, mix_coeffs [2,C] -> (mixed_up, mixed_gate), each [T,B,C] (the inputs of
    linear_up and linear_gate)."""
    _check_act("x", x, 3)
    if tuple(mix.shape) != (NE, x.shape[-1]):
        raise ValueError(f"mix must be [2,C] = {(NE, x.shape[-1])}, got {tuple(mix.shape)}")
    if x.shape[-1] % 8:
        raise NotImplementedError("C must be a multiple of 8")
    return _lib.native().cmix_lerp(x, mix)


def _n_check(*ts):
    for t in ts:
        if t.device.type != "cuda" or t.dtype != torch.bfloat16:
            raise TypeError("channel-mix epilogues take bfloat16 CUDA tensors")
        if t.shape != ts[0].shape:
            raise ValueError("operand shapes differ")
    if ts[0].numel() % 8:
        raise NotImplementedError("element count must be a multiple of 8")


def relu_sq(up: torch.Tensor) -> torch.Tensor:
    """square(relu(up)) (rwkv6_layer_specs.py:524), bf16 in and out, fp32 inside."""
    _n_check(up)
    return _lib.native().relu_sq(up)


def sigmoid_gate(out: torch.Tensor, gate_pre: torch.Tensor) -> torch.Tensor:
    """out * sigmoid(gate_pre) (rwkv6_layer_specs.py:533-536), bf16 in and out."""
    _n_check(out, gate_pre)
    return _lib.native().sigmoid_gate(out, gate_pre)
