"""Dense attention forward on MI355X (the callee for additional keys/values and for
kernel_size == input size).  Counterpart of the forward half of the reference's
src/natten/backends/blackwell_fmha.py:190-260, including sequence-packed variable-length batches."""

from __future__ import annotations

from typing import Optional, Tuple, Union

import torch
from torch import Tensor

from . import _lib, torch_ops
from .checks import fmha_tensor_checks
from .fna import SUPPORTED_DTYPES, is_fp8, pad_head_dim, resolve_scale
from .tile_config import padded_head_dim, takes_narrow_rows


def amd_fmha(
    query: Tensor, key: Tensor, value: Tensor, is_causal: bool = False, scale: Optional[float] = None,
    return_lse: bool = False,
    q_scale=None,
    k_scale=None,
    v_scale=None,
    out_dtype: Optional[torch.dtype] = None,
    cumulative_seqlen_Q: Optional[Tensor] = None,
    cumulative_seqlen_KV: Optional[Tensor] = None,
    max_seqlen_Q: int = 0,
    max_seqlen_KV: int = 0,
) -> Union[Tensor, Tuple[Tensor, Tensor]]:
    """8-bit float operands are widened to bf16 (exactly) and multiplied in bf16; `q_scale`,
    `k_scale`, `v_scale` (number or per-head tensor) are their dequantisation scales.
    `out_dtype` defaults to the dtype of `query`.  With `cumulative_seqlen_{Q,KV}` (validated by
    the caller) the operands are sequence-packed (batch = 1) and every sequence attends to its
    own keys only."""
    fmha_tensor_checks(query, key, value, must_match_head_dims=True)
    if not query.is_cuda:
        raise NotImplementedError(f"natten_amd runs on MI355X device tensors only; got a tensor on {query.device}.")
    if query.dtype not in SUPPORTED_DTYPES:
        raise NotImplementedError(f"natten_amd attention supports {SUPPORTED_DTYPES}, got {query.dtype}.")
    head_dim = query.shape[-1]
    if head_dim > 128 or head_dim % 8 != 0:
        raise NotImplementedError(f"natten_amd attention supports head_dim <= 128, multiple of 8; got {head_dim}.")
    if is_fp8(query.dtype) and head_dim % 16 != 0:
        raise NotImplementedError(f"natten_amd attention needs head_dim % 16 == 0 for 8-bit floats; got {head_dim}.")
    scale = scale or head_dim**-0.5
    d_pad = padded_head_dim(head_dim)
    if torch.is_grad_enabled() and (query.requires_grad or key.requires_grad or value.requires_grad):
        if is_fp8(query.dtype):
            raise NotImplementedError("natten_amd attention has no backward pass for 8-bit float operands.")
        if cumulative_seqlen_Q is not None:
            out, lse = AmdFmhaVarlenFunction.apply(
                query, key, value, bool(is_causal), float(scale), cumulative_seqlen_Q, cumulative_seqlen_KV,
                int(max_seqlen_Q), int(max_seqlen_KV),
            )
        else:
            out, lse = AmdFmhaFunction.apply(query, key, value, bool(is_causal), float(scale))
        if out_dtype is not None and out.dtype != out_dtype:
            out = out.to(out_dtype)
        return (out, lse) if return_lse else out
    if d_pad != head_dim and cumulative_seqlen_Q is None and takes_narrow_rows(head_dim, query.dtype):
        d_pad = head_dim
    q, k, v = query.contiguous(), key.contiguous(), value.contiguous()
    if d_pad != head_dim:
        q, k, v = (pad_head_dim(t, d_pad).contiguous() for t in (q, k, v))
    if is_fp8(query.dtype):
        # a one-token tile with no dilation is the identity permutation: a plain widening copy
        q, k, v = (torch_ops.token_permute(t, (1,), (1,), True, widen=True) for t in (q, k, v))
    scales = dict(
        q_scale=resolve_scale(q_scale, q.shape[-2], q.device, "q_scale"),
        k_scale=resolve_scale(k_scale, k.shape[-2], q.device, "k_scale"),
        v_scale=resolve_scale(v_scale, k.shape[-2], q.device, "v_scale"),
    )
    if cumulative_seqlen_Q is not None:
        if max_seqlen_Q == 0 or max_seqlen_KV == 0:
            # every sequence is empty on one side: nothing attends to anything
            out = torch.zeros_like(q)
            lse = torch.full(q.shape[:-1], float("-inf"), dtype=torch.float32, device=q.device)
        else:
            out, lse = torch_ops.attention_forward_varlen(
                q, k, v, cumulative_seqlen_Q.contiguous(), cumulative_seqlen_KV.contiguous(), max_seqlen_Q,
                max_seqlen_KV, bool(is_causal), scale, **scales,
            )
    else:
        out, lse = torch_ops.attention_forward(q, k, v, bool(is_causal), scale, **scales)
    if d_pad != head_dim:
        out = out[..., :head_dim].contiguous()
    out_dtype = out_dtype or query.dtype
    if out.dtype != out_dtype:
        out = out.to(out_dtype)
    if return_lse:
        return out, lse
    return out


class AmdFmhaFunction(torch.autograd.Function):
    """Dense attention with a backward pass (fp16 / bf16, fixed-length batches): the backward
    kernels of neighborhood attention on the 1-D problem whose window is the whole key sequence.
    Counterpart of the reference's
    src/natten/backends/blackwell_fmha.py:52-170; the gradient of LSE is not propagated.  The saved
    output and LSE are the returned tensors themselves (see AmdFnaFunction)."""

    @staticmethod
    def forward(ctx, query, key, value, is_causal, scale):
        with torch.no_grad():
            out, lse = amd_fmha(query, key, value, is_causal=is_causal, scale=scale, return_lse=True)
        ctx.save_for_backward(query, key, value, out, lse)
        ctx.args = (is_causal, scale)
        ctx.mark_non_differentiable(lse)
        ctx.set_materialize_grads(False)
        return out, lse

    @staticmethod
    def backward(ctx, d_out, d_lse):
        query, key, value, out, lse = ctx.saved_tensors
        if d_out is None:  # (what came after the output passed no gradient on)
            return (torch.zeros_like(query), torch.zeros_like(key), torch.zeros_like(value)) + (None,) * 2
        is_causal, scale = ctx.args
        head_dim = query.shape[-1]
        d_pad = padded_head_dim(head_dim)
        query, key, value, out, d_out = (
            pad_head_dim(t.contiguous(), d_pad).contiguous() for t in (query, key, value, out, d_out)
        )
        dq, dk, dv = torch_ops.attention_backward(query, key, value, out, d_out, lse.contiguous(), is_causal, scale)
        if d_pad != head_dim:
            dq, dk, dv = (t[..., :head_dim] for t in (dq, dk, dv))
        return dq, dk, dv, None, None


class AmdFmhaVarlenFunction(torch.autograd.Function):
    """Variable-length dense attention with a backward pass, both on the packed operands as they are: one
    set of launches for all sequences.  Counterpart of the varlen arguments of
    src/natten/backends/blackwell_fmha.py:52-170."""

    @staticmethod
    def forward(ctx, query, key, value, is_causal, scale, cu_q, cu_kv, max_q, max_kv):
        with torch.no_grad():
            out, lse = amd_fmha(query, key, value, is_causal=is_causal, scale=scale, return_lse=True,
                                cumulative_seqlen_Q=cu_q, cumulative_seqlen_KV=cu_kv, max_seqlen_Q=max_q,
                                max_seqlen_KV=max_kv)
        ctx.save_for_backward(query, key, value, out, lse, cu_q, cu_kv)
        ctx.args = (is_causal, scale)
        ctx.max_seqlens = (int(max_q), int(max_kv))
        ctx.mark_non_differentiable(lse)
        ctx.set_materialize_grads(False)
        return out, lse

    @staticmethod
    def backward(ctx, d_out, d_lse):
        query, key, value, out, lse, cu_q, cu_kv = ctx.saved_tensors
        is_causal, scale = ctx.args
        head_dim = query.shape[-1]
        max_q, max_kv = ctx.max_seqlens
        if d_out is None or max_q == 0 or max_kv == 0 or query.shape[1] == 0 or key.shape[1] == 0:
            # what came after the output passed no gradient on, or no sequence has both queries and keys: the
            # output does not depend on the operands
            return (torch.zeros_like(query), torch.zeros_like(key), torch.zeros_like(value)) + (None,) * 6
        d_pad = padded_head_dim(head_dim)
        q, k, v, o, do = (pad_head_dim(t.contiguous(), d_pad).contiguous() for t in (query, key, value, out, d_out))
        dq, dk, dv = torch_ops.attention_backward_varlen(
            q, k, v, o, do, lse.contiguous(), cu_q.to(torch.int32).contiguous(), cu_kv.to(torch.int32).contiguous(), is_causal,
            scale, max_q,
        )
        if d_pad != head_dim:
            dq, dk, dv = (t[..., :head_dim] for t in (dq, dk, dv))
        return (dq, dk, dv) + (None,) * 6
