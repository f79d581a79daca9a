"""Drop-in for fla's RWKV-6 ops, backed by the HIP kernels of librwkv6_amd.so.

The reference calls ``fused_recurrent_rwkv6(r, k, v, w, u, scale=1.)[0]`` at
/root/reference/rwkv_megatron/rwkv6_layer_specs.py:339 after laying its
tensors out head-first (:333-337).  fla also exports ``chunk_rwkv6`` with the
same contract (4th argument named ``g``).  Both names are provided here:

    o, final_state = chunk_rwkv6(r, k, v, g, u, scale=None, initial_state=None,
                                 output_final_state=False)

* r, k, g(=w): [B,H,T,K]; v: [B,H,T,V]; u: [H,K]; K == V == 64.
* g / w is LOG-space decay (the caller passes ``-exp(decay)``, :336).
* scale None or -1 means K**-0.5 (fla's convention); any other float is used as is.
* initial_state: [B,H,K,V] (computed in fp32); final_state is fp32 or None.
* o has r's dtype.  Arithmetic: bf16 operands on MFMA, fp32 accumulation and fp32
  carried state.  bf16 r, k, v, g are used as they are; fp32 / fp16 ones are rounded to
  bf16 on entry (one rounding each, 2^-9 relative), so an fp32 caller gets bf16-operand
  arithmetic, not fp32 arithmetic.  u is used in its own dtype (fp32 or bf16).
* The autograd function is csrc/autograd.cpp's.  Backward returns gradients for r, k, v, g, u and initial_state, and accepts a
  gradient on final_state.
"""
from __future__ import annotations

import torch

from . import _lib

_HEAD = 64


def _validate(r, k, v, w, u, initial_state):
    for name, t in (("r", r), ("k", k), ("v", v), ("w", w), ("u", u)):
        if not isinstance(t, torch.Tensor):
            raise TypeError(f"{name} must be a torch.Tensor")
        if t.device.type != "cuda":
            raise ValueError(f"{name} must live on the GPU (got {t.device})")
        if t.dtype not in (torch.bfloat16, torch.float16, torch.float32):
            raise TypeError(f"{name}: unsupported dtype {t.dtype}")
    if r.dim() != 4:
        raise ValueError(f"r must be [B,H,T,K], got shape {tuple(r.shape)}")
    B, H, T, K = r.shape
    if k.shape != r.shape or w.shape != r.shape:
        raise ValueError(f"k and w must match r's shape {tuple(r.shape)}")
    if v.dim() != 4 or v.shape[:3] != r.shape[:3]:
        raise ValueError(f"v must be [B,H,T,V] with B,H,T of r, got {tuple(v.shape)}")
    V = v.shape[-1]
    if u.shape != (H, K):
        raise ValueError(f"u must be [H,K] = {(H, K)}, got {tuple(u.shape)}")
    if K != _HEAD or V != _HEAD:
        raise NotImplementedError(f"head size must be K == V == {_HEAD}, got K={K}, V={V}")
    if initial_state is not None and tuple(initial_state.shape) != (B, H, K, V):
        raise ValueError(f"initial_state must be [B,H,K,V] = {(B, H, K, V)}")
    devs = {t.device for t in (r, k, v, w, u)}
    if initial_state is not None:
        devs.add(initial_state.device)
    if len(devs) != 1:
        raise ValueError("all tensors must be on the same device")


def chunk_rwkv6(r, k, v, g, u, scale=None, initial_state=None, output_final_state=False,
                checkpoint_level=None, cu_seqlens=None, head_first=True):
    """RWKV-6 WKV, fla ``chunk_rwkv6`` contract.  Returns ``(o, final_state or None)``."""
    if cu_seqlens is not None:
        raise NotImplementedError("variable-length batches (cu_seqlens) are not supported")
    if not head_first:
        raise NotImplementedError("only the head-first [B,H,T,K] layout is supported")
    if scale is None or scale == -1:
        scale = _HEAD ** -0.5
    scale = float(scale)
    try:
        out = _lib.native().wkv6(r, k, v, g, u, initial_state, scale, bool(output_final_state))
    except TypeError:                       # not a tensor: say which; or raised on the way (a hook)
        _validate(r, k, v, g, u, initial_state)
        raise
    if out is None:                         # an argument does not fit: say which
        _validate(r, k, v, g, u, initial_state)
        raise ValueError("WKV6 arguments do not fit together")
    return out


def fused_recurrent_rwkv6(r, k, v, w, u, scale=-1, initial_state=None, output_final_state=False,
                          causal=True, cu_seqlens=None, head_first=True):
    """RWKV-6 WKV, fla ``fused_recurrent_rwkv6`` contract (the name the reference imports at
    rwkv6_layer_specs.py:47 and calls at :339).  Same kernels as ``chunk_rwkv6``."""
    if not causal:
        raise NotImplementedError("only causal RWKV-6 is defined")
    return chunk_rwkv6(r, k, v, w, u, scale=scale, initial_state=initial_state,
                       output_final_state=output_final_state, cu_seqlens=cu_seqlens,
                       head_first=head_first)


def wkv6_seqfirst(r, k, v, decay, u, num_heads, scale=1.0, initial_state=None,
                  output_final_state=False):
    """WKV6 for the time-mix module: r, k, v, decay [T,B,H*64] (decay before -exp) ->
    (o [B,H,T,64] head-first, final_state or None).  Same arithmetic as chunk_rwkv6 with
    w = -exp(decay)."""
    for name, t in (("r", r), ("k", k), ("v", v), ("decay", decay)):
        if not isinstance(t, torch.Tensor) or t.device.type != "cuda":
            raise ValueError(f"{name} must be a CUDA tensor")
        if t.dim() != 3 or t.shape != r.shape:
            raise ValueError(f"{name} must be [T,B,C] like r, got {tuple(t.shape)}")
    T, B, C = r.shape
    if C % num_heads or C // num_heads != _HEAD:
        raise NotImplementedError(f"head size must be {_HEAD} (C={C}, heads={num_heads})")
    if tuple(u.shape) != (num_heads, _HEAD):
        raise ValueError(f"u must be [H,64], got {tuple(u.shape)}")
    if initial_state is not None and tuple(initial_state.shape) != (B, num_heads, _HEAD, _HEAD):
        raise ValueError("initial_state must be [B,H,64,64]")
    return _lib.native().wkv6_seqfirst(r, k, v, decay, u, initial_state, float(scale), int(num_heads),
                                       bool(output_final_state))
