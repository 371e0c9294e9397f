"""The linear maps of a neighborhood attention layer on kernels of their own (csrc/linear.hpp).

A layer's step was bound by everything around its attention: on 4 x 56 x 56 tokens, H 8, D 32, 7 x 7, bf16, 410 us of device time
of which 101 were the attention's kernels, the rest being library products that do not split their long contractions
(143 us for two weight gradients), reductions of the bias gradients (44), and nine strided copies of queries, keys,
values and their gradients (47), each a launch that the host makes (some thirty a step).  Here the map writes queries, keys
and values as the attention takes them, its backward reads their gradients as the attention returns them, bias gradients come with
the weight gradients, and the step is one autograd node of nine launches."""

from __future__ import annotations

import functools
from typing import Optional, Tuple

import torch
from torch import Tensor, nn
from torch.autograd import forward_ad
from torch.nn.modules.module import _has_any_global_hook

from . import _lib, torch_ops
from .checks import check_args_against_input
from .fna import amd_fna_generic, backward_route
from .functional import neighborhood_attention_generic
from .tile_config import BACKWARD_TILE_SIZE, choose_tile_shapes

# Widest layer that takes these kernels: where measuring against the library ended, not where the library was found to be the
# faster way (us, here / there: 12544 tokens, 256 -> 768: y 13.7 / 21.7, dx 10.0 / 18.6, dw and db 20.5 / 90; 36864
# tokens, 512 -> 1536: y 79.6 / 104, dx level (64.3 / 60 to 65), dw and db 108 / 254; 196 tokens, 512 -> 1536: y 7.9 / 18.9,
# dx 12.6 / 18.2, dw and db 11.1 / 27; below 20 us a call is the time the host takes to make it).
MAX_COLUMNS = 512


def _plain(t: Optional[Tensor], dtype: torch.dtype, device: torch.device, align: int) -> bool:
    return (type(t) in (Tensor, nn.Parameter) and t.dtype == dtype and t.device == device and t.is_contiguous()
            and t.data_ptr() % align == 0)


def _nothing_watches() -> bool:
    """No tracer, transform or mode is active that looks at the operators a layer calls."""
    return not (torch_ops._tracing() or torch.jit.is_tracing() or torch.is_autocast_enabled("cuda")
                or torch._C._len_torch_dispatch_stack() or torch._C._len_torch_function_stack()
                or torch._C._functorch.peek_interpreter_stack() is not None or forward_ad._current_level >= 0)


def takes_linear(module: nn.Module, x: Tensor, parts: int) -> bool:
    """Whether the kernels stand for calling `module` on x [.., columns] and splitting the result into `parts` of as
    many columns each: a plain nn.Linear of these sizes that nothing is attached to, 16-bit operands on one device, columns
    that the kernels take, and no one watching the call.  Everything else goes the way of nn.Linear.  (Who watches is
    asked first: a tracer cannot take a data pointer apart, a transform's tensors have none.)"""
    return _nothing_watches() and _fits(module, x, parts)


def _fits(module: nn.Module, x: Tensor, parts: int) -> bool:
    if type(module) is not nn.Linear or "forward" in module.__dict__:
        return False
    if module._forward_hooks or module._forward_pre_hooks or module._backward_hooks or module._backward_pre_hooks or _has_any_global_hook():
        return False
    n, k = module.out_features, module.in_features
    if k != x.shape[-1] or n != parts * k:  # (another output width than the layer's, or a map that does not fit)
        return False
    if k % 64 or k > MAX_COLUMNS:
        return False
    if type(x) not in (Tensor, nn.Parameter) or not x.is_cuda or x.dtype not in (torch.float16, torch.bfloat16):
        return False
    if not 0 < x.numel() < 2**31 * 64 or x.numel() // k >= 2**31 - 128 or x.data_ptr() % 16:
        return False
    w, b = module.weight, module.bias
    return (_plain(w, x.dtype, x.device, 16) and w.shape == (n, k)
            and (b is None or (_plain(b, x.dtype, x.device, 8) and b.shape == (n,))))


def _aligned(t: Tensor) -> Tensor:
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


class _Linear(torch.autograd.Function):
    """x [.., *in columns] -> `parts` tensors of `shape`: x w^T + b with its columns split into that many."""

    @staticmethod
    def forward(ctx, x, weight, bias, parts, shape):
        ctx.save_for_backward(x, weight)
        ctx.has_bias = bias is not None
        return _lib.linear_forward(x, weight, bias, parts, shape)

    @staticmethod
    def backward(ctx, *d_outs):
        x, weight = ctx.saved_tensors
        n, k = weight.shape
        if torch.is_grad_enabled():  # (a graph of the backward itself is wanted: in operations that have one)
            dy = torch.cat([d.reshape(-1, n // len(d_outs)) for d in d_outs], dim=1)
            dx = (dy @ weight).reshape(x.shape) if ctx.needs_input_grad[0] else None
            dw = dy.t() @ x.reshape(-1, k) if ctx.needs_input_grad[1] else None
            db = dy.sum(0) if ctx.has_bias and ctx.needs_input_grad[2] else None
            return dx, dw, db, None, None
        d_outs = [_aligned(d) for d in d_outs]
        return (*_lib.linear_backward(d_outs, x, weight, *ctx.needs_input_grad[:2], ctx.has_bias and ctx.needs_input_grad[2]),
                None, None)


@functools.lru_cache(maxsize=1024)
def _layer_backward_plan(layout, heads, head_dim, kernel_size, stride, dilation, is_causal):
    """Tile shapes of the attention's backward launches on the original tensors, or None where a layer's step is not one
    autograd node: whole-input windows (dense attention), padded head dims, layouts that the launches take permuted."""
    if head_dim not in (32, 64, 128) or (len(layout) == 1 and kernel_size[0] == layout[0]):
        return None
    if all(k == x and not c for x, k, c in zip(layout, kernel_size, is_causal)):
        return None
    problem = (layout, kernel_size, stride, dilation, is_causal)
    pair = choose_tile_shapes(*problem, BACKWARD_TILE_SIZE, BACKWARD_TILE_SIZE)
    fused, tiles, role = backward_route(*problem, heads * head_dim * 2, *pair)
    return (*tiles, *role) if fused else None


def _layer_nodes(x, w_qkv, b_qkv, w_proj, b_proj, heads, problem, scale):
    """A layer as three autograd nodes: map, attention, map."""
    shape = (*x.shape[:-1], heads, x.shape[-1] // heads)
    q, k, v = _Linear.apply(x, w_qkv, b_qkv, 3, shape)
    out = neighborhood_attention_generic(q, k, v, *problem, scale=scale)
    return _Linear.apply(out, w_proj, b_proj, 1, x.shape)[0]


class _Layer(torch.autograd.Function):
    """A layer's step as one node: between three of them the engine hands each gradient over from Python to Python
    (4 x 56 x 56 tokens, H 8, D 32, 7 x 7: 373 us a step as three nodes, 267 as one)."""

    @staticmethod
    def forward(ctx, x, w_qkv, b_qkv, w_proj, b_proj, heads, problem, scale, plan):
        q, k, v = _lib.linear_forward(x, w_qkv, b_qkv, 3, (*x.shape[:-1], heads, x.shape[-1] // heads))
        out, lse = amd_fna_generic(q, k, v, *problem, scale, return_lse=True, run_persistent_kernel=None, _checked=True)
        ctx.save_for_backward(x, w_qkv, b_qkv, w_proj, b_proj, q, k, v, out, lse)
        ctx.args = (heads, problem, scale, plan)
        return _lib.linear_forward(out, w_proj, b_proj, 1, x.shape)[0]

    @staticmethod
    def backward(ctx, d_out):
        x, w_qkv, b_qkv, w_proj, b_proj, q, k, v, out, lse = ctx.saved_tensors
        heads, problem, scale, plan = ctx.args
        need_x, need_w1, need_b1, need_w2, need_b2 = ctx.needs_input_grad[:5]
        if torch.is_grad_enabled():  # (a graph of the backward itself is wanted)
            leaves = (x, w_qkv, b_qkv, w_proj, b_proj)
            wanted = [t for t, need in zip(leaves, ctx.needs_input_grad) if need]
            grads = iter(torch.autograd.grad(_layer_nodes(*leaves, heads, problem, scale), wanted, d_out, create_graph=True))
            return (*(next(grads) if need else None for need in ctx.needs_input_grad[:5]), None, None, None, None)
        d_out = _aligned(d_out)
        dx = dw1 = db1 = None
        first = need_x or need_w1 or need_b1
        d_attn, dw2, db2 = _lib.linear_backward((d_out,), out, w_proj, first, need_w2, need_b2)
        if first:
            grads = _lib.fna_backward_fused(q, k, v, d_attn, lse, None, *problem, scale, *plan, out=out)
            dx, dw1, db1 = _lib.linear_backward(grads, x, w_qkv, need_x, need_w1, need_b1)
        return dx, dw1, db1, dw2, db2, None, None, None, None


def layer_step(qkv: nn.Linear, proj: nn.Linear, x: Tensor, heads: int, problem, scale: float) -> Optional[Tensor]:
    """proj(attention(qkv(x))), or None where the maps or their surroundings are not what takes_linear takes.  `problem`:
    kernel size, stride, dilation and causality per dimension."""
    if not (takes_linear(qkv, x, 3) and _fits(proj, x, 1)):
        return None
    params = (qkv.weight, qkv.bias, proj.weight, proj.bias)
    layout, head_dim = tuple(x.shape[1:-1]), x.shape[-1] // heads
    x = x.contiguous()
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, *params)):
        check_args_against_input(x.unsqueeze(-1), *problem)
        plan = _layer_backward_plan(layout, heads, head_dim, *problem)
        if plan is None:
            return _layer_nodes(x, *params, heads, problem, scale)
        return _Layer.apply(x, *params, heads, problem, scale, plan)
    q, k, v = _lib.linear_forward(x, qkv.weight, qkv.bias, 3, (*x.shape[:-1], heads, head_dim))
    out = neighborhood_attention_generic(q, k, v, *problem, scale=scale)
    return _lib.linear_forward(out, proj.weight, proj.bias, 1, x.shape)[0]
