"""Float32 forward on the original tensors (boxes of 16 queries, blocks of 16 keys) where its boxes and
rows can go wrong: extents below a block, remainders, groups of unequal length, every head dim class,
against the float64 oracle at the bar of tests/test_gpu_fp32.py, and against the token-permuted kernel."""

import pytest
import torch

from natten_amd.functional import na1d, na2d, na3d
from tests.gpu_utils import assert_close, oracle_full, to_np
from tests.test_gpu_fp32 import ATOL32, make

pytestmark = pytest.mark.gpu

NA = {1: na1d, 2: na2d, 3: na3d}

CASES = [
    # B, shape, H, Hkv, D, kernel, stride, dilation, causal
    (1, (2,), 1, 1, 8, (2,), (1,), (1,), (False,)),
    (3, (17,), 2, 1, 24, (3,), (3,), (5,), (True,)),
    (1, (257,), 3, 3, 128, (64,), (64,), (1,), (False,)),
    (2, (3, 50), 2, 2, 120, (2, 17), (2, 5), (1, 2), (True, False)),
    (1, (33, 5), 4, 2, 72, (31, 3), (16, 1), (1, 1), (False, True)),
    (1, (16, 16), 1, 1, 64, (13, 13), (1, 1), (1, 1), (False, False)),
    (1, (3, 4, 37), 2, 1, 56, (2, 3, 9), (1, 3, 2), (1, 1, 4), (False, True, False)),
    (2, (11, 6, 5), 1, 1, 96, (5, 2, 3), (4, 2, 1), (2, 3, 1), (True, True, True)),
    (1, (20, 9, 8), 2, 2, 32, (20, 9, 8), (1, 1, 1), (1, 1, 1), (True, False, False)),
]


@pytest.mark.parametrize("case", CASES)
def test_boxes_and_rows(case):
    B, shape, H, Hkv, D, kernel, stride, dilation, causal = case
    q, k, v = make(B, shape, H, Hkv, D, seed=sum(shape) + D)
    na = NA[len(shape)]
    out, lse = na(q, k, v, kernel, stride=stride, dilation=dilation, is_causal=causal, return_lse=True)
    ref_o, ref_l = oracle_full(q, k, v, kernel, stride, dilation, causal)
    assert_close("out", to_np(out), ref_o, atol=ATOL32, rtol=ATOL32)
    assert_close("lse", to_np(lse), ref_l, atol=ATOL32, rtol=ATOL32)
    # the permuted kernel (reached by fixing tiles) sums the same products in another order
    tiles = {1: ((128,), (64,)), 2: ((8, 16), (8, 8)), 3: ((2, 8, 8), (4, 4, 4))}[len(shape)]
    out_p, lse_p = na(q, k, v, kernel, stride=stride, dilation=dilation, is_causal=causal, return_lse=True,
                      q_tile_shape=tiles[0], kv_tile_shape=tiles[1])
    assert_close("out", to_np(out), to_np(out_p), atol=ATOL32, rtol=ATOL32)
    assert_close("lse", to_np(lse), to_np(lse_p), atol=ATOL32, rtol=ATOL32)


def test_operands_that_are_not_sixteen_byte_aligned():
    q, k, v = make(1, (100,), 2, 2, 32, seed=1)
    shifted = [torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for t in (q, k, v)]
    assert any(t.data_ptr() % 16 for t in shifted)
    assert torch.equal(na1d(*shifted, 9), na1d(q, k, v, 9))


def test_large_logits_and_infinite_rows():
    # logits that outgrow the running maximum from block to block, and a query all of whose logits are -inf
    q, k, v = make(1, (64,), 1, 1, 32, seed=2)
    k = k * torch.linspace(1, 200, 64, device="cuda").view(1, 64, 1, 1)
    out, lse = na1d(q, k, v, 33, return_lse=True)
    ref_o, ref_l = oracle_full(q, k, v, (33,), (1,), (1,), (False,))
    # (logits reach 1e3: their float32 rounding, 2^-24 of that per term, appears in the exponent)
    assert_close("out", to_np(out), ref_o, atol=2e-3, rtol=2e-3)
    assert_close("lse", to_np(lse), ref_l, atol=2e-3, rtol=1e-5)
    q[:, 5], k[:] = 0.0, 1.0
    q[:, 5, :, 0], k[..., 0] = 1.0, -float("inf")
    out, lse = na1d(q, k, v, 33, return_lse=True)
    assert torch.equal(out[0, 5, 0], torch.zeros(32, device="cuda")) and lse[0, 5, 0] == -float("inf")


def test_lse_of_long_windows_is_rounded_not_biased():
    # windows of 1025 keys, values between 4 and 8.5: the rounding of the result and of the term added last are
    # up to 2^-22 / sqrt(12) = 1.4e-7 rms each, 2e-7 together, and the logits' own errors average out over a window.
    # (The logarithm of the whole sum, whose maximum may lag, was low by 2.6e-7 in the mean and 4.1e-7 rms.)
    q, k, v = make(2, (2048,), 2, 2, 32, seed=3)
    _, lse = na1d(q, k, v, 1025, stride=64, return_lse=True)
    _, ref = oracle_full(q, k, v, (1025,), (64,), (1,), (False,))
    error = to_np(lse).astype("float64") - ref
    assert 4 < ref.min() and ref.max() < 8.5
    assert abs(error.mean()) < 1e-7 and (error**2).mean() ** 0.5 < 3e-7
