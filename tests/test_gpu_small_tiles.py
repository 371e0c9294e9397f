"""The 64 x 64 tile pair that the one-launch forward takes for small windows, and launch layouts with few
groups of Q tiles per XCD, against the CPU oracle; where the pair is chosen (CPU)."""

import pytest
import torch

from natten_amd.fna import _open_call_plan
from natten_amd.functional import na1d, na2d, na3d
from natten_amd.tile_config import choose_small_forward_tiles, choose_tile_shapes
from tests.gpu_utils import assert_close, make_qkv, oracle_full, to_np

NA = {1: na1d, 2: na2d, 3: na3d}

CASES = [
    # shape, kernel, stride, dilation, causal, D
    ((40, 33), (7, 7), (1, 1), (1, 1), (False, False), 64),
    ((66, 66), (4, 36), (1, 2), (1, 1), (False, True), 64),       # 2 groups of unequal length per head before evening out
    ((37, 44), (8, 11), (2, 1), (2, 1), (True, False), 32),       # groups of 19 and 18 rows, causal along them
    ((10, 19, 21), (3, 5, 5), (1, 1, 2), (1, 1, 1), (False, True, False), 24),
    ((3000,), (196,), (8,), (1,), (False,), 32),
]


def chosen(shape, kernel, stride, dilation, causal):
    big = choose_tile_shapes(shape, kernel, stride, dilation, causal, 128, 64, anchored=True)
    return choose_small_forward_tiles(shape, kernel, stride, dilation, causal, *big)


@pytest.mark.parametrize("case", CASES)
def test_the_cases_below_take_the_pair(case):
    assert chosen(*case[:5]) is not None


def test_a_launch_kind_given_keeps_the_larger_pair():
    # True and False promise each other's bits, hence tiles; None is free to take others
    args = ((64, 64), (13, 13), (1, 1), (1, 1), (False, False))
    plan = {kind: _open_call_plan(torch.bfloat16, (2, 64, 64, 8, 64), 8, *args[1:], kind) for kind in (None, False, True)}
    large = choose_tile_shapes(*args, 128, 64, anchored=True)
    assert plan[None][:2] == chosen(*args) and plan[None][:2] != large
    assert plan[False] == (*large, False, 1) and plan[True] == (*large, True, 1)


def test_where_the_pair_is_chosen():
    assert chosen((64, 64), (13, 13), (1, 1), (1, 1), (False, False)) is not None
    assert chosen((64, 64), (48, 48), (1, 1), (1, 1), (False, False)) is None       # hardly fewer pairs
    assert chosen((4096,), (33,), (1,), (1,), (False,)) is None                     # two tiles a workgroup
    assert chosen((64, 3), (7, 3), (1, 1), (1, 1), (False, False)) is None or chosen(
        (64, 3), (7, 3), (1, 1), (1, 1), (False, False))[1][1] <= 3                 # no group narrower than a key tile


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, dtype):
    shape, kernel, stride, dilation, causal, D = case
    q, k, v = make_qkv(2, shape, 4, 2, D, dtype, seed=3)
    with torch.no_grad():
        out, lse = NA[len(shape)](q, k, v, kernel, stride=stride, dilation=dilation, is_causal=causal, return_lse=True)
    ref_o, ref_l = oracle_full(q, k, v, kernel, stride, dilation, causal)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)


@pytest.mark.gpu
def test_launch_kinds_given_agree_bit_for_bit():
    q, k, v = make_qkv(2, (40, 33), 4, 2, 64, torch.bfloat16, seed=5)
    with torch.no_grad():
        queue, plain, left_open = (na2d(q, k, v, (7, 7), run_persistent_kernel=kind, return_lse=True) for kind in (True, False, None))
    assert all(torch.equal(a, b) for a, b in zip(queue, plain))
    for a, b in zip(left_open, plain):  # (other tiles: other sums of the same windows)
        assert_close("tiles left open", to_np(a), to_np(b))
