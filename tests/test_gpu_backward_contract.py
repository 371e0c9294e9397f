"""The backward entry points of the C library by their argument lists: the neighborhood ones take the
forward's LSE and rowsum(d_out * out) as they are, and what natten_amd_backward_prepare wrote only where
`roles` says so.  Gradients against the float64 oracle at the tolerance of the backward tests."""

import ctypes

import numpy as np
import pytest
import torch

from natten_amd import _lib
from natten_amd.fna import amd_fna_generic
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np

SHAPE, KERNEL, STRIDE, DILATION, CAUSAL = (16, 24), (7, 9), (1, 2), (1, 1), (False, True)
TILE = (8, 16)


def problem(D, dtype):
    gen = torch.Generator().manual_seed(D)
    q, d_out = (torch.randn((2, *SHAPE, 4, D), generator=gen).to(dtype).cuda() for _ in range(2))
    k, v = (torch.randn((2, *SHAPE, 2, D), generator=gen).to(dtype).cuda() for _ in range(2))
    out, lse = amd_fna_generic(q, k, v, KERNEL, STRIDE, DILATION, CAUSAL, return_lse=True)
    return q, k, v, d_out, out, lse


def i32(values):
    return (ctypes.c_int32 * len(values))(*[int(x) for x in values])


def head_major(x):
    return x.flatten(1, 2).transpose(1, 2).contiguous()


def fused(q, k, v, d_out, lse, delta, q_scaled, calls):
    grads = [torch.full_like(t, float("nan")) for t in (q, k, v)]
    for roles in calls:
        rc = _lib.lib().natten_amd_fna_backward_fused(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), d_out.data_ptr(), lse.data_ptr(), delta.data_ptr(),
            *(g.data_ptr() for g in grads), q_scaled.data_ptr(), _lib.DTYPE_CODES[q.dtype], 2, q.shape[0], q.shape[3], k.shape[3],
            q.shape[4], i32(SHAPE), i32(KERNEL), i32(STRIDE), i32(DILATION), i32(CAUSAL), i32(TILE), i32(TILE), q.shape[4] ** -0.5,
            roles, torch.cuda.current_stream().cuda_stream)
        assert rc == 0, _lib.lib().natten_amd_last_error()
    return grads


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_lse_and_delta_as_they_are_or_prepared(D, dtype):
    q, k, v, d_out, out, lse = problem(D, dtype)
    delta = _lib.compute_delta(out, d_out)
    ref = O.na_backward(*(to_np(t) for t in (q, k, v, d_out)), KERNEL, STRIDE, DILATION, CAUSAL)
    plain = (head_major(lse), head_major(delta), torch.empty_like(q))
    q_scaled = torch.empty_like(q)
    neg_delta, neg_lse2 = _lib.backward_prepare(q, out, d_out, lse, D**-0.5, q_scaled)
    prepared = (neg_lse2, neg_delta, q_scaled)
    for args, calls in ((plain, (3,)), (plain, (2, 1)), (prepared, (7,)), (prepared, (6, 5))):
        for name, g, r in zip(("dq", "dk", "dv"), fused(q, k, v, d_out, *args, calls), ref):
            assert_close(f"{name}, roles {calls}", to_np(g), r, atol=2e-2, rtol=2e-2)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 128])
def test_permuted_operands_take_lse_and_delta_as_they_are(D):
    q, k, v, d_out, out, lse = problem(D, torch.bfloat16)
    delta = _lib.compute_delta(out, d_out)
    perm = lambda x: _lib.token_permute(x.contiguous(), TILE, DILATION, True)
    qp, kp, vp, dop = (perm(t) for t in (q, k, v, d_out))
    lse_p, delta_p = (perm(t.unsqueeze(-1)).squeeze(-1).transpose(1, 2).contiguous() for t in (lse, delta))
    padded = (16, 32)
    grads = [torch.empty_like(t) for t in (qp, kp, vp)]
    rc = _lib.lib().natten_amd_fna_backward(
        qp.data_ptr(), kp.data_ptr(), vp.data_ptr(), dop.data_ptr(), lse_p.data_ptr(), delta_p.data_ptr(),
        *(g.data_ptr() for g in grads), grads[0].data_ptr(), _lib.DTYPE_CODES[q.dtype], 2, qp.shape[0], qp.shape[1], kp.shape[1],
        qp.shape[2], kp.shape[2], D, i32(padded), i32(padded), i32(SHAPE), i32(KERNEL), i32(STRIDE), i32(DILATION), i32(CAUSAL),
        i32(TILE), i32(TILE), D**-0.5, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.lib().natten_amd_last_error()
    ref = O.na_backward(*(to_np(t) for t in (q, k, v, d_out)), KERNEL, STRIDE, DILATION, CAUSAL)
    for name, g, r in zip(("dq", "dk", "dv"), grads, ref):
        back = _lib.token_unpermute(g, SHAPE, TILE, DILATION, True)
        assert_close(name, to_np(back), r, atol=2e-2, rtol=2e-2)


def test_lse_and_delta_cost_a_copy_each():
    from torch.utils._python_dispatch import TorchDispatchMode

    class Launches(TorchDispatchMode):
        count = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            if not func.is_view and "view" not in func.name():
                Launches.count += 1
            return out

    lse, delta = torch.randn(2, 5, 7, 3), torch.randn(2, 5, 7, 3)
    with Launches():
        a, b = _lib._head_major(lse, delta)
    assert Launches.count <= 2
    np.testing.assert_array_equal(a.numpy(), lse.reshape(2, 35, 3).transpose(1, 2).numpy())
    np.testing.assert_array_equal(b.numpy(), delta.reshape(2, 35, 3).transpose(1, 2).numpy())
