"""Public operations: attention, na1d, na2d, na3d.

Mirrors the reference's src/natten/functional.py (attention :74-348,
neighborhood_attention_generic :354-564, na1d/na2d/na3d :567-1151): same signatures, same
argument rules and error classes, same self-attention fast path and additional-KV merge.
There is one backend (the MI355X kernels); the reference's NVIDIA-only performance arguments are
accepted and ignored, except `q_tile_shape` / `kv_tile_shape`, which select the kernel's tiles.
"""

from __future__ import annotations

import functools
import math
from typing import Dict, Optional, Tuple, Union

import torch
from torch import Tensor

from .attn_merge import merge_attentions
from .checks import (
    additional_kv_tensor_checks,
    check_all_args,
    check_args_against_input,
    fmha_tensor_checks,
    is_self_attention,
    na_tensor_checks,
)
from .fmha import amd_fmha
from .fna import amd_fna_generic, amd_fna_with_context, is_fp8
from .utils.varlen import varlen_tensor_checks

_BACKEND_FNA = "amd-fna"
_BACKEND_FMHA = "amd-fmha"


def attention(
    query: Tensor,
    key: Tensor,
    value: Tensor,
    is_causal: bool = False,
    scale: Optional[float] = None,
    # varlen parameters
    seqlens_Q: Optional[Tensor] = None,
    seqlens_KV: Optional[Tensor] = None,
    cumulative_seqlen_Q: Optional[Tensor] = None,
    cumulative_seqlen_KV: Optional[Tensor] = None,
    max_seqlen_Q: Optional[int] = None,
    max_seqlen_KV: Optional[int] = None,
    # backend parameters
    backend: Optional[str] = None,
    q_tile_size: Optional[int] = None,
    kv_tile_size: Optional[int] = None,
    backward_q_tile_size: Optional[int] = None,
    backward_kv_tile_size: Optional[int] = None,
    backward_kv_splits: Optional[int] = None,
    backward_use_pt_reduction: bool = False,
    run_persistent_kernel: Optional[bool] = None,
    kernel_schedule=None,
    torch_compile: bool = False,
    return_lse: bool = False,
    # quantised (8-bit float) operands; not in the reference
    q_scale=None,
    k_scale=None,
    v_scale=None,
    out_dtype: Optional[torch.dtype] = None,
) -> Union[Tensor, Tuple[Tensor, Tensor]]:
    """Dot product attention on `[batch, seqlen, heads, head_dim]` tensors (heads last).

    `is_causal` is top-left aligned.  Variable-length batches use the sequence-packed layout
    (batch = 1, sequences back to back): pass either `seqlens_Q` / `seqlens_KV` (int32 device
    tensors; costs a synchronisation) or `cumulative_seqlen_{Q,KV}` and `max_seqlen_{Q,KV}` from
    `natten_amd.utils.varlen.generate_varlen_parameters`
    (reference: src/natten/functional.py:74-348).  Returns the output, and the float32 logsumexp
    `[batch, seqlen, heads]` when `return_lse=True`.  For e4m3 / e5m2 operands `q_scale`, `k_scale`,
    `v_scale` (number or per-head tensor) are the dequantisation scales and `out_dtype` the
    result type (default: the operands' type, as in the reference).

    Results are the same from call to call.  From a batch of two on, where the last workgroups would leave most
    of the chip idle, their key walks are split and the parts summed in float: the entries of such a batch
    may then differ from each other, and from a call on one entry alone, in the order of summation (by
    about one rounding of the result).  Batches of one and packed sequences are never split: those give each
    other's bits.
    """
    fmha_tensor_checks(query, key, value, must_match_head_dims=True)
    cumulative_seqlen_Q, cumulative_seqlen_KV, max_seqlen_Q, max_seqlen_KV = varlen_tensor_checks(
        query, key, value, seqlens_Q=seqlens_Q, seqlens_KV=seqlens_KV, cumulative_seqlen_Q=cumulative_seqlen_Q,
        cumulative_seqlen_KV=cumulative_seqlen_KV, max_seqlen_Q=max_seqlen_Q, max_seqlen_KV=max_seqlen_KV,
    )
    if backend not in (None, _BACKEND_FMHA):
        raise NotImplementedError(f"Unrecognized attention backend {backend}; natten_amd provides '{_BACKEND_FMHA}'.")
    return amd_fmha(
        query, key, value, is_causal=is_causal, scale=scale, return_lse=return_lse,
        q_scale=q_scale, k_scale=k_scale, v_scale=v_scale, out_dtype=out_dtype,
        cumulative_seqlen_Q=cumulative_seqlen_Q, cumulative_seqlen_KV=cumulative_seqlen_KV,
        max_seqlen_Q=max_seqlen_Q, max_seqlen_KV=max_seqlen_KV,
    )


def neighborhood_attention_generic(
    query: Tensor,
    key: Tensor,
    value: Tensor,
    kernel_size,
    stride=1,
    dilation=1,
    is_causal=False,
    scale: Optional[float] = None,
    additional_keys: Optional[Tensor] = None,
    additional_values: Optional[Tensor] = None,
    attention_kwargs: Optional[Dict] = None,
    # Perf-related args
    backend: Optional[str] = None,
    q_tile_shape=None,
    kv_tile_shape=None,
    backward_q_tile_shape=None,
    backward_kv_tile_shape=None,
    backward_kv_splits=None,
    backward_use_pt_reduction: bool = False,
    run_persistent_kernel: Optional[bool] = None,
    kernel_schedule=None,
    torch_compile: bool = False,
    return_lse: bool = False,
    q_scale=None,
    k_scale=None,
    v_scale=None,
    out_dtype: Optional[torch.dtype] = None,
    fp8_matmul: Optional[bool] = None,
) -> Union[Tensor, Tuple[Tensor, Tensor]]:
    na_tensor_checks(query, key, value)
    additional_kv_tensor_checks(query, key, value, additional_keys, additional_values)
    na_dim = query.dim() - 3
    kernel_size, stride, dilation, is_causal = check_all_args(na_dim, kernel_size, stride, dilation, is_causal)
    check_args_against_input(query, kernel_size=kernel_size, stride=stride, dilation=dilation, is_causal=is_causal)
    if backend not in (None, _BACKEND_FNA):
        raise NotImplementedError(f"Unrecognized backend {backend}; natten_amd provides '{_BACKEND_FNA}'.")

    has_additional_attention = additional_keys is not None and additional_values is not None
    if has_additional_attention and query.dtype == torch.float32:
        # refused before anything is launched: the additional context goes through dense attention
        raise NotImplementedError(
            "natten_amd: float32 operands with additional_keys / additional_values are not supported (dense "
            "attention, which serves the additional context, has no float32 kernel); use fp16 or bf16 operands."
        )
    attn_kwargs = dict(attention_kwargs or {})
    attn_kwargs.pop("torch_compile", None)

    # (float32 operands stay with the neighborhood kernel, which has a float32 form; dense attention has none)
    if query.dtype != torch.float32 and is_self_attention(query, kernel_size=kernel_size, is_causal=is_causal,
                                                          has_additional_attention=has_additional_attention):
        # a window covering the whole input is plain attention over the flattened tokens
        query_shape = query.shape
        q = query.flatten(1, na_dim)
        k = key.flatten(1, na_dim)
        v = value.flatten(1, na_dim)
        if has_additional_attention:
            k = torch.cat([k, additional_keys], dim=1)
            v = torch.cat([v, additional_values], dim=1)
        out, lse = attention(
            q, k, v, is_causal=is_causal[0], scale=scale, return_lse=True,
            q_scale=q_scale, k_scale=k_scale, v_scale=v_scale, out_dtype=out_dtype, **attn_kwargs,
        )
        lse_shape = list(query_shape[:-1])
        out = out.reshape(*lse_shape, v.shape[-1])
        lse = lse.reshape(*lse_shape)
        return (out, lse) if return_lse else out

    scale = scale or query.shape[-1] ** -0.5
    final_dtype = out_dtype or query.dtype
    # Partial results before a merge: bf16 for 8-bit float operands; the operands' own type when
    # gradients are wanted (the merge's backward writes the merged output and LSE into the very
    # tensors the partial attentions saved, so those must reach it uncast); else the final type.
    needs_grad = torch.is_grad_enabled() and any(
        t is not None and t.requires_grad for t in (query, key, value, additional_keys, additional_values)
    )
    if (has_additional_attention and not needs_grad and not attn_kwargs and q_tile_shape is None and kv_tile_shape is None
            and q_scale is None and k_scale is None and v_scale is None and final_dtype == query.dtype):
        # one launch over the window and the context, where there is one (it rounds to the operands' type: a caller
        # who asks for float32 gets the merge's, and one who asks for what the merge does not take its refusal)
        joint = amd_fna_with_context(query, key, value, additional_keys, additional_values, kernel_size, stride, dilation,
                                     is_causal, scale, run_persistent_kernel)
        if joint is not None:
            return joint if return_lse else joint[0]
    if is_fp8(query.dtype):
        work_dtype = torch.bfloat16
    else:
        work_dtype = query.dtype if needs_grad else final_dtype
    output, lse = amd_fna_generic(
        query, key, value, kernel_size=kernel_size, stride=stride, dilation=dilation, is_causal=is_causal,
        scale=scale, q_tile_shape=q_tile_shape, kv_tile_shape=kv_tile_shape, return_lse=True,
        q_scale=q_scale, k_scale=k_scale, v_scale=v_scale,
        out_dtype=work_dtype if has_additional_attention else final_dtype, fp8_matmul=fp8_matmul,
        backward_q_tile_shape=backward_q_tile_shape, backward_kv_tile_shape=backward_kv_tile_shape,
        run_persistent_kernel=run_persistent_kernel, _checked=True,
    )

    if has_additional_attention:
        # the additional keys / values share the dequantisation scales of key / value
        add_out, add_lse = attention(
            query.flatten(1, na_dim), additional_keys, additional_values, is_causal=False, scale=scale,
            return_lse=True, q_scale=q_scale, k_scale=k_scale, v_scale=v_scale, out_dtype=work_dtype, **attn_kwargs,
        )
        merged_out, merged_lse = merge_attentions(
            [output.flatten(1, na_dim), add_out], [lse.flatten(1, na_dim), add_lse]
        )
        output = merged_out.reshape(output.shape).to(final_dtype)
        lse = merged_lse.reshape(output.shape[:-1])

    return (output, lse) if return_lse else output


def _use_work_queue(run_persistent_kernel: Optional[bool], is_causal, num_q_tiles: int = 1 << 30,
                    kv_tiles_per_q_tile: int = 1 << 10) -> bool:
    """`run_persistent_kernel` as given, or the measured default.  The work-queue launch (resident
    workgroups pull Q tiles from per-XCD queues; a workgroup fetches its next position between its last
    KV tile and its stores) saves the 3-4 us a CU slot stands empty between two workgroups of a
    one-workgroup-per-tile launch: 2.5-10 % on the large shapes measured, causal or not; on 2 048 Q
    tiles x 16 KV tiles (c3) the two are within 2 % of each other either way, and below that the queue's
    bookkeeping costs more than it saves.  `num_q_tiles`: Q tiles over all batch entries, dilation
    groups and heads; `kv_tiles_per_q_tile`: KV tiles a Q tile visits (an estimate).  True
    and False give the same bits (without KV splits); None leaves the tile shapes open as well."""
    if run_persistent_kernel is not None:
        return bool(run_persistent_kernel)
    return num_q_tiles >= 2048 and num_q_tiles * kv_tiles_per_q_tile >= 65536


@torch.compiler.assume_constant_result  # (plain Python on launch constants: not for the tracer to look into)
def work_queue_default(batch: int, heads: int, token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape,
                       kv_tile_shape) -> bool:
    """The launch kind the ops pick when `run_persistent_kernel` is None, from the problem's tile counts."""
    return _work_queue_default(int(batch), int(heads), *(tuple(x) for x in (
        token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape)))


@functools.lru_cache(maxsize=1024)
def _work_queue_default(batch, heads, token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape):
    tiles = batch * heads
    for X, d, qt in zip(token_layout, dilation, q_tile_shape):
        tiles *= -(-(-(-X // d)) // qt) * d
    return _use_work_queue(None, is_causal, tiles, _kv_tiles_per_q_tile(
        token_layout, kernel_size, stride, dilation, q_tile_shape, kv_tile_shape))


def _kv_tiles_per_q_tile(token_layout, kernel_size, stride, dilation, q_tile_shape, kv_tile_shape) -> int:
    """KV tiles a Q tile visits at most (causal masks and borders visit fewer)."""
    visits = 1
    for X, k, s, d, qt, kt in zip(token_layout, kernel_size, stride, dilation, q_tile_shape, kv_tile_shape):
        # keys the queries of one Q tile attend along this dimension: a window per stride group the tile spans
        visits *= -(-min(-(-X // d), k + (-(-qt // s) - 1) * s) // kt)
    return visits


@torch.compiler.assume_constant_result
def kv_splits_default(batch: int, heads: int, token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape,
                      kv_tile_shape) -> int:
    """How many workgroups share the KV tiles of a Q tile when `kv_splits` is None: 4 or 2 when the
    problem has so few Q tiles that, split, they still leave every workgroup a compute unit of its
    own (256 of them) and every split has at least four KV tiles of every Q tile; else 1.  Measured
    (split kernel + the 6-7 us merge launch against the unsplit kernel, microseconds): 64 Q tiles of
    34 KV tiles 28 + 6 two ways and 22 + 7 four ways against 46; a 64 x 64 image with 2 heads and a
    33 x 33 window 33 + 6 and 24 + 7 against 58; 256 Q tiles of 34 KV tiles two ways 46 + 6 against
    53 (no gain: the loop only shortens in proportion while a workgroup does not share its SIMDs)."""
    return _kv_splits_default(int(batch), int(heads), *(tuple(x) for x in (
        token_layout, kernel_size, dilation, is_causal, q_tile_shape, kv_tile_shape)))


@torch.compiler.assume_constant_result
def narrow_kv_splits_default(batch: int, heads: int, token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape,
                             kv_tile_shape) -> int:
    """kv_splits_default for rows between the native head dims, whose single launch has no padded copies beside it:
    split from 24 KV tiles a Q tile on.  The device is faster split at any length (60 random problems), but a call
    takes the host 30 us split and 20 in one launch, and up to there the one launch is over by then.  Measured
    (one launch / split and merged, device us, bf16): 10 tiles, 4096 tokens, D 48 17.2 / 16.3; 18 tiles, 2048 tokens,
    H 8, D 96 29.8 / 26.6; 27 tiles, 9 x 27 x 12, D 56 36.5 / 27.2; 34 tiles, 8192 tokens, D 96 44.3 / 26.4; 81 tiles, 16 x
    32 x 32, D 96 114.6 / 68.6."""
    if _kv_tiles_per_q_tile(token_layout, kernel_size, stride, dilation, q_tile_shape, kv_tile_shape) < 24:
        return 1
    return kv_splits_default(batch, heads, token_layout, kernel_size, stride, dilation, is_causal, q_tile_shape, kv_tile_shape)


def paired_groups_default(batch: int, heads: int, head_dim: int, token_layout, kernel_size, stride, dilation, is_causal,
                          q_tile_shape, kv_tile_shape, splits: int = 1, small: bool = False) -> bool:
    """Whether a forward launch has two groups of waves in the workgroup of a Q tile: where every Q tile (128 x 64 tokens) has a
    compute unit of its own, and its KV tiles are enough to pay for the sums' way through LDS.  One group /
    two, us, bf16, by KV tiles of a Q tile, 256 Q tiles each.  Head dim 128: 6 14.1 / 14.8, 10 17.8 / 18.0
    (in two dimensions, most of them with a mask, 20.3 / 19.5), 18 25.4 / 25.2 (30.7 / 28.0), 34 41.9 / 40.5, 66 71.5 / 68.1; head
    dim 64: 6 11.4 / 10.9, 10 12.8 / 12.0, 34 27.8 / 24.2.  `splits`: what kv_splits_default says.  A walk that two workgroups
    would share is that of a pair up to 24 KV tiles at head dim 64 and 16 at 128: no merge launch, which also takes
    the host 26 us a call (split and merged / paired, device: 12 tiles, 64 Q tiles 13.8 / 12.5 and 17.3 / 17.4, 128 Q tiles
    15.0 / 12.7 and 20.6 / 17.8; 20 tiles 17.3 / 16.1 and 24.9 / 25.5; 34 tiles 21.4 / 21.8 and 30.0 / 30.9).  (Without
    masks at head dim 128 the entry point takes one group, faster still.)  `small`: tiles of 64 x 64 tokens are
    the alternative (choose_small_forward_tiles), which up to 128 Q tiles of 128 leave each a compute unit as well: 64 x 64, 15 x 15,
    H 4 13.0 / 13.9, 33 x 47, 19 x 19, H 6 18.0 / 18.6; 256 Q tiles: 128 x 128, 13 x 13, H 2 14.3 / 12.8, 21 x 21 22.3 / 17.9."""
    if splits > 2 or head_dim not in (64, 128) or math.prod(q_tile_shape) != 128 or math.prod(kv_tile_shape) != 64:
        return False
    if any(x // d < t for x, d, t in zip(token_layout, dilation, kv_tile_shape)):
        return False  # (groups narrower than a tile have an instance of their own)
    visits = _kv_tiles_per_q_tile(token_layout, kernel_size, stride, dilation, q_tile_shape, kv_tile_shape)
    if splits == 2:
        return visits <= (24 if head_dim == 64 else 16)
    tiles = batch * heads
    for X, d, qt in zip(token_layout, dilation, q_tile_shape):
        tiles *= -(-(-(-X // d)) // qt) * d
    return (128 if small else 0) < tiles <= 256 and visits >= (8 if head_dim == 64 else 16)


@functools.lru_cache(maxsize=1024)
def _kv_splits_default(batch, heads, token_layout, kernel_size, dilation, is_causal, q_tile_shape, kv_tile_shape):
    tiles, min_visits = batch * heads, 1
    for X, k, d, c, qt, kt in zip(token_layout, kernel_size, dilation, is_causal, q_tile_shape, kv_tile_shape):
        extent = -(-X // d)
        tiles *= -(-extent // qt) * d
        # fewest KV tiles a Q tile meets along this dimension: a whole window, or one key where causal
        min_visits *= max((1 if c else min(extent, k)) // kt, 1)
    for splits in (4, 2):
        if tiles * splits <= 256 and min_visits >= 4 * splits:
            return splits
    return 1


def _make_na(na_dim: int, name: str):
    def op(
        query: Tensor,
        key: Tensor,
        value: Tensor,
        kernel_size,
        stride=1,
        dilation=1,
        is_causal=False,
        scale: Optional[float] = None,
        additional_keys: Optional[Tensor] = None,
        additional_values: Optional[Tensor] = None,
        attention_kwargs: Optional[Dict] = None,
        backend: Optional[str] = None,
        q_tile_shape=None,
        kv_tile_shape=None,
        backward_q_tile_shape=None,
        backward_kv_tile_shape=None,
        backward_kv_splits=None,
        backward_use_pt_reduction: bool = False,
        run_persistent_kernel: Optional[bool] = None,
        kernel_schedule=None,
        torch_compile: bool = False,
        return_lse: bool = False,
        q_scale=None,
        k_scale=None,
        v_scale=None,
        out_dtype: Optional[torch.dtype] = None,
        fp8_matmul: Optional[bool] = None,
    ) -> Union[Tensor, Tuple[Tensor, Tensor]]:
        if query.dim() != na_dim + 3:
            raise ValueError(
                f"{name} expects rank-{na_dim + 3} tensors [batch, {'*' if na_dim > 1 else ''}tokens, heads, head_dim], "
                f"got rank {query.dim()}."
            )
        return neighborhood_attention_generic(
            query=query, key=key, value=value, kernel_size=kernel_size, stride=stride, dilation=dilation,
            is_causal=is_causal, scale=scale, additional_keys=additional_keys, additional_values=additional_values,
            attention_kwargs=attention_kwargs, backend=backend, q_tile_shape=q_tile_shape,
            kv_tile_shape=kv_tile_shape, backward_q_tile_shape=backward_q_tile_shape,
            backward_kv_tile_shape=backward_kv_tile_shape, backward_kv_splits=backward_kv_splits,
            backward_use_pt_reduction=backward_use_pt_reduction, run_persistent_kernel=run_persistent_kernel,
            kernel_schedule=kernel_schedule, torch_compile=torch_compile, return_lse=return_lse,
            q_scale=q_scale, k_scale=k_scale, v_scale=v_scale, out_dtype=out_dtype, fp8_matmul=fp8_matmul,
        )

    op.__name__ = name
    op.__qualname__ = name
    op.__doc__ = (
        f"{na_dim}-D neighborhood attention on heads-last tensors "
        f"`[batch, {', '.join('XYZ'[:na_dim])}, heads, head_dim]`.\n\n"
        "kernel_size, stride, dilation: int or tuple per dimension (kernel_size >= 2, stride <= kernel_size, "
        "kernel_size * dilation <= input size); is_causal: bool or tuple.  additional_keys / additional_values "
        "`[batch, seqlen, heads_kv, head_dim]` add context every query attends to.  Returns the output and, with "
        "`return_lse=True`, the float32 logsumexp `[batch, *tokens, heads]`.  For e4m3 / e5m2 operands `q_scale`, "
        "`k_scale`, `v_scale` (number or per-head tensor) are the dequantisation scales, `out_dtype` the result "
        "type (default: the operands' type) and `fp8_matmul=False` trades the 8-bit matrix instruction for "
        "bf16 products on exactly widened operands (slower, more accurate)."
    )
    return op


na1d = _make_na(1, "na1d")
na2d = _make_na(2, "na2d")
na3d = _make_na(3, "na3d")

__all__ = ["attention", "na1d", "na2d", "na3d", "neighborhood_attention_generic"]
