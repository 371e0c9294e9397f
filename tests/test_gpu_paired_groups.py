"""GPU: forward launches with two groups of waves per Q tile: even and odd numbers of KV tiles, one tile, walks longer than are
described at once, tiles at the edges of groups; against the CPU oracle, and where the launch is chosen (CPU)."""

import pytest
import torch

from natten_amd import _lib
from natten_amd.fna import _open_call_plan
from natten_amd.functional import na1d
from tests.gpu_utils import make_qkv, sampled_check

CASES = [
    # shape, kernel, stride, dilation, causal, tiles
    ((700,), (64,), (64,), (1,), (False,), ((128,), (64,))),                                  # two or three tiles
    ((333,), (3,), (1,), (1,), (True,), ((128,), (64,))),                                     # a second group with one tile
    ((300,), (2,), (2,), (2,), (False,), ((128,), (64,))),                                    # ... or none of its own
    ((9000,), (8200,), (8,), (1,), (False,), ((128,), (64,))),                                # 65 and more each
    ((41, 53), (17, 20), (1, 3), (1, 1), (False, True), ((8, 16), (8, 8))),
    ((60, 47), (13, 9), (1, 1), (2, 3), (True, False), ((16, 8), (4, 16))),
    ((9, 17, 21), (5, 7, 8), (1, 2, 1), (1, 1, 2), (True, False, False), ((2, 8, 8), (4, 4, 4))),
    ((16, 32, 32), (8, 16, 16), (4, 8, 8), (1, 1, 1), (False, False, False), ((2, 8, 8), (1, 8, 8))),  # nearly no masks
    # the same with queries past the end (without, a launch of head dim 128 takes the kernel of one group)
    ((16, 32, 30), (8, 16, 16), (4, 8, 8), (1, 1, 1), (False, False, False), ((2, 8, 8), (1, 8, 8))),
]


def test_cases_that_need_no_mask():
    # (at head dim 128 these run in one group)
    assert [i for i, (*problem, tiles) in enumerate(CASES) if _lib.fully_block_sparse(*problem, *tiles)] == [7]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, head_dim, dtype):
    shape, kernel, stride, dilation, causal, tiles = case
    q, k, v = make_qkv(2, shape, 2, 1, head_dim, dtype, seed=11)
    out, lse = _lib.fna_forward_fused_paired(q, k, v, kernel, stride, dilation, causal, head_dim**-0.5, *tiles)
    sampled_check(q, k, v, out, lse, kernel, stride, dilation, causal, 300, seed=1)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("case", CASES)
def test_infinite_values_reach_the_queries_that_one_group_lets_them_reach(case, head_dim):
    # (an odd walk's middle tile lies before both groups: the second multiplies its values by probabilities of zero)
    shape, kernel, stride, dilation, causal, tiles = case
    q, k, v = make_qkv(2, shape, 2, 2, head_dim, torch.bfloat16, seed=12)
    tokens = v.view(2, -1, 2, head_dim)
    gen = torch.Generator().manual_seed(3)
    for b in range(2):
        for h in range(2):
            # every batch entry and head has infinities of its own: few, many
            tokens[b, torch.randperm(tokens.shape[1], generator=gen)[: (2, 5, 20, 80)[2 * b + h]].cuda(), h, 7] = float("inf")
    problem = (q, k, v, kernel, stride, dilation, causal, head_dim**-0.5, *tiles)
    ref, ref_lse = _lib.fna_forward_fused(*problem)
    out, lse = _lib.fna_forward_fused_paired(*problem)
    assert torch.isinf(ref).any() and not torch.isnan(lse).any()
    assert torch.equal(torch.isnan(out), torch.isnan(ref)) and torch.equal(torch.isinf(out), torch.isinf(ref))


@pytest.mark.gpu
def test_chosen_call_replays_in_a_graph():
    q, k, v = make_qkv(1, (8192,), 4, 2, 64, torch.bfloat16, seed=2)
    with torch.no_grad():
        ref, ref_lse = na1d(q, k, v, 1024, return_lse=True)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out, lse = na1d(q, k, v, 1024, return_lse=True)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, ref) and torch.equal(lse, ref_lse)
    sampled_check(q, k, v, ref, ref_lse, (1024,), (1,), (1,), (False,), 300, seed=1)


def test_where_it_is_chosen():
    def kind(shape, heads, head_dim, kernel, launch=None, dtype=torch.bfloat16):
        ones = (1,) * len(shape)
        return _open_call_plan(dtype, (1, *shape, heads, head_dim), heads, kernel, ones, ones, (False,) * len(shape), launch)[2]

    assert kind((32768,), 1, 128, (2048,)) == "paired" and kind((32768,), 1, 64, (512,)) == "paired"
    assert kind((32768,), 2, 128, (2048,)) is False        # more Q tiles than compute units
    assert kind((32768,), 1, 128, (512,)) is False         # few KV tiles
    assert kind((8192,), 1, 128, (2048,)) is False         # a split launch
    assert kind((32768,), 1, 96, (2048,)) is False
    assert kind((128, 128), 2, 64, (13, 13)) == "paired" and kind((64, 64), 4, 64, (15, 15)) is False  # 64 x 64 tiles: 256 and fewer
    assert kind((8192,), 2, 64, (600,)) == "paired" and kind((8192,), 2, 64, (3500,)) is False   # a two-way split's walks: short ones
    assert kind((32768,), 1, 128, (2048,), launch=False) is False and kind((32768,), 1, 128, (2048,), launch=True) is True
