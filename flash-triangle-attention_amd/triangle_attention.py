"""The AlphaFold2 triangle self-attention block (Alg. 13 "starting node", Alg. 14 "ending node")
around attention(): layer norm, the q/k/v/bias/gate projections of the pair representation z,
the fused attention, sigmoid gating and the output projection.

    blk = TriangleAttention(c_z=128, c_hidden=32, n_heads=4, starting=True).cuda()
    out = blk(z)                      # z: (B, L, L, c_z) -> (B, L, L, c_z)

The attention runs in fp16, or in bf16 when z is bf16.  `dropout_p` drops attention weights while the
module is in training mode; every call draws a fresh mask seed from torch's CPU generator (so layers
and steps differ and torch.manual_seed reproduces a run), or takes the `seed` passed to forward().

What the block does NOT do around the kernels: no permute copies.  The projections write
(B, L, L, H*D); attention() reads q, k, v as (B, H, L, L, D) *views* of that (strides passed through
to the kernels), and the ending-node variant works on the L1<->L2 transposed view of z.  Only the
bias, (B, L, L, H) -> (B, H, L, L), is laid out contiguously (2 bytes per pair and head).

Upstream has no such block (its README shows the op only); the input recipe of its AF2-shaped use,
z -> projections -> (B, H, L, L, D), is what this file packages.  `reference_forward` is the same
block with the naive O(L^3) attention, used by the tests.
"""
from __future__ import annotations

import math

import torch
from torch import nn
from torch.nn.modules.module import _has_any_global_hook
from torch.overrides import _get_current_function_mode_stack
from torch.utils._device import DeviceContext

import fta_lib
from flash_tt_attn import _attention, attention, reference_tt_attn

__all__ = ["TriangleAttention"]

# Added to the bias of padded key positions: its exponent underflows to exactly 0 in fp16 and fp32
# (attention() also takes -inf there; a finite value keeps the naive reference free of inf - inf).
_KEY_MASK_BIAS = -30000.0


# Submodules in the order in which the fused path takes their weights, and whether it takes a bias with them.
_SUBMODULES = (("layer_norm", nn.LayerNorm, True), ("linear_q", nn.Linear, False), ("linear_k", nn.Linear, False),
               ("linear_v", nn.Linear, False), ("linear_b", nn.Linear, False), ("linear_g", nn.Linear, True),
               ("linear_o", nn.Linear, True))


def _function_mode_on() -> bool:
    """Whether a mode sees or rewrites the calls of torch functions (torch.device as a context or the default device is
    one, too, but only says where new tensors go)."""
    return torch._C._len_torch_function_stack() > 0 and any(type(m) is not DeviceContext for m in _get_current_function_mode_stack())


class TriangleAttention(nn.Module):
    def __init__(self, c_z: int, c_hidden: int = 32, n_heads: int = 4, starting: bool = True, dropout_p: float = 0.0):
        super().__init__()
        self.c_z, self.c_hidden, self.n_heads, self.starting = c_z, c_hidden, n_heads, starting
        self.dropout_p = float(dropout_p)
        hd = c_hidden * n_heads
        self.layer_norm = nn.LayerNorm(c_z)
        self.linear_q = nn.Linear(c_z, hd, bias=False)
        self.linear_k = nn.Linear(c_z, hd, bias=False)
        self.linear_v = nn.Linear(c_z, hd, bias=False)
        self.linear_b = nn.Linear(c_z, n_heads, bias=False)
        self.linear_g = nn.Linear(c_z, hd)
        self.linear_o = nn.Linear(hd, c_z)

    def _operands(self, z, key_mask):
        """q, k, v as (B, H, L, L, D) 16-bit views, bias as (B, H, L, L) of the same type, the gate, all from z."""
        if not self.starting:
            z = z.transpose(1, 2)
        B, L1, L2, _ = z.shape
        H, D = self.n_heads, self.c_hidden
        x = self.layer_norm(z)
        op = torch.bfloat16 if z.dtype == torch.bfloat16 else torch.float16
        split = lambda t: t.to(op).view(B, L1, L2, H, D).permute(0, 3, 1, 2, 4)
        q, k, v = split(self.linear_q(x)), split(self.linear_k(x)), split(self.linear_v(x))
        # b[j, k] of the pair (j, k), shared by every row i: (B, L, L, H) -> (B, H, L, L)
        bias = self.linear_b(x).permute(0, 3, 1, 2)
        if key_mask is not None:  # (B, L): 0 marks padded positions, which no query may attend to
            bias = bias + (key_mask.to(bias.dtype)[:, None, None, :] - 1.0) * (-_KEY_MASK_BIAS)
        bias = bias.to(op).contiguous()
        gate = torch.sigmoid(self.linear_g(x))
        return q, k, v, bias, gate

    def _finish(self, o, gate, dtype):
        B, H, L1, L2, D = o.shape
        o = o.permute(0, 2, 3, 1, 4).reshape(B, L1, L2, H * D).to(gate.dtype)
        out = self.linear_o(gate * o).to(dtype)
        return out if self.starting else out.transpose(1, 2)

    def _fused(self, z, key_mask, seed):
        """The whole block in the kernels of csrc/fta_block.hip (three launches forward, eight backward), for
        plain fp16, bf16 or fp32 modules of the sizes built there (c_z and n_heads * c_hidden of 64 or 128);
        None where this does not apply: other sizes, autocast, mixed types, a call that something traces,
        sees through a mode or transforms, hooked, parametrised, wrapped or replaced submodules, a subclass."""
        if type(self) is not TriangleAttention or not z.is_cuda or _has_any_global_hook() or _function_mode_on():
            return None
        native = fta_lib.native()
        if native is None:
            return None
        weights, modules = [], self._modules
        for name, kind, has_bias in _SUBMODULES:
            m = modules.get(name)
            if type(m) is not kind:
                return None
            d = m.__dict__
            if d["_forward_hooks"] or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]:
                return None
            own = d["_parameters"]
            # (a forward of the instance's own, as wrappers put there; a weight or bias that is no parameter any more)
            if "forward" in d or "weight" not in own or "bias" not in own:
                return None
            weights.append(own["weight"])
            if has_bias:
                weights.append(own["bias"])
            elif own["bias"] is not None:
                return None
        norm = modules["layer_norm"]
        if norm.normalized_shape != (z.shape[-1],):
            return None
        scope = _attention.forward.__globals__  # (the module that holds the PRECISE_BACKWARD switch)
        p = self.dropout_p if self.training else 0.0
        try:
            return native.block(z, key_mask, weights, self.n_heads, self.c_hidden, self.starting, norm.eps, p,
                                seed if p > 0.0 else 0, scope)  # (no seed: one is drawn if the call is taken)
        except TypeError:  # (a seed beyond 63 bits)
            return None

    def forward(self, z: torch.Tensor, key_mask: torch.Tensor | None = None, seed: int | None = None) -> torch.Tensor:
        out = self._fused(z, key_mask, seed)
        if out is not None:
            return out
        q, k, v, bias, gate = self._operands(z, key_mask)
        sm = 1.0 / math.sqrt(self.c_hidden)
        if self.training and self.dropout_p > 0.0:
            o = attention(q, k, v, bias, sm, self.dropout_p) if seed is None else attention(q, k, v, bias, sm, self.dropout_p, seed)
        else:
            o = attention(q, k, v, bias, sm)
        return self._finish(o, gate, z.dtype)

    def reference_forward(self, z: torch.Tensor, key_mask: torch.Tensor | None = None) -> torch.Tensor:
        """Same block, naive attention in fp32 on the same 16-bit-rounded operands (any device), no dropout."""
        q, k, v, bias, gate = self._operands(z, key_mask)
        o = reference_tt_attn(q.float(), k.float(), v.float(), bias.float(), 1.0 / math.sqrt(self.c_hidden))
        return self._finish(o, gate, z.dtype)
