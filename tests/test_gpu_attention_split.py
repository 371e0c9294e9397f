"""Dense attention whose last round of workgroups, or only one, is split over the keys: query and key counts around tiles, all
head dims, GQA, causal; against the CPU oracle and the unsplit launch.  What the plan splits (CPU)."""

import numpy as np
import pytest
import torch

import natten_amd
from natten_amd import _lib
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np


def rand(shape, dtype, seed):
    return torch.randn(shape, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()


def test_plan():
    plan = lambda *a: _lib.attention_split_plan(0, *a)
    assert plan(2, 1000, 4000, 4, 128, False)[1] > 1          # 64 Q tiles on the whole chip
    assert plan(2, 1000, 1000, 4, 128, False) == (0, 1)        # over before a second launch is made
    assert plan(1, 1000, 4000, 8, 128, False) == (0, 1)        # one sequence: the bits of a packed call
    assert plan(2, 4096, 4096, 16, 64, False) == (0, 1)        # whole rounds
    assert plan(2, 8200, 512, 16, 64, False) == (0, 1)         # too few keys
    assert plan(2, 9000, 9000, 24, 64, True) == (0, 1)         # causal: rounds even out
    positions, splits = plan(2, 4097, 4097, 16, 64, False)     # a third round of 32 Q tiles
    assert positions % 8 == 0 and 32 <= positions < 64 and 2 <= splits <= 16
    for args in ((2, 1000, 4000, 4, 128, False), (3, 1700, 5000, 5, 64, False), (2, 3600, 3600, 2, 96, True)):
        positions, splits = plan(*args)
        tiles = -(-args[1] // 128) * args[0] * args[3]
        assert splits > 1 and positions >= tiles % 512 and tiles % 512 * splits <= 512


def test_plan_where_the_one_launch_holds_three_waves():
    """Head dim 32, and head dim 64 without masks: the split launch holds two waves per SIMD at either."""
    plan = lambda *a: _lib.attention_split_plan(0, *a)
    for S, H in ((2560, 16), (3072, 12), (5120, 8), (4096, 17)):    # 576 .. 1088 Q tiles: 768 fit one round
        assert plan(2, S, S, H, 64, False) == (0, 1)
    assert plan(2, 8448, 3072, 4, 64, False)[1] > 1 and plan(2, 9216, 9216, 4, 64, False)[1] > 1   # long walks, few left over
    assert plan(2, 2560, 4001, 16, 64, False)[1] > 1                # masks: two waves either way
    for S, H in ((4097, 16), (3500, 16), (4097, 12), (10000, 10)):
        assert plan(2, S, S, H, 32, False) == (0, 1)
    assert plan(2, 12547, 12547, 4, 32, False)[1] > 1
    for S, H in ((4000, 4), (8000, 2), (4000, 3), (4000, 2)):       # one round
        positions, splits = plan(2, S, S, H, 32, False)
        assert splits > 1 and 2 * H * -(-S // 128) * splits <= 512


def test_plan_counts_by_xcd():
    """The XCD with the most Q tiles ends a launch: where the shares are uneven, no XCD keeps more than whole rounds unsplit."""
    plan = lambda *a: _lib.attention_split_plan(0, *a)
    assert plan(5, 3100, 3100, 5, 128, False) == (0, 1)     # 91 tiles on some: two halves of the last 27 save too little
    assert plan(3, 5000, 5000, 9, 128, False) == (96, 5)    # 140 on some: the last 12 of each
    assert plan(2, 8257, 3001, 8, 128, False)[0] == 32      # 132 on every other one
    assert plan(2, 6500, 6500, 6, 96, False) == (112, 4)
    assert plan(3, 3522, 3522, 3, 128, False) == (0, 1)     # 35 of 64: not twice


def test_plan_counts_positions_without_a_q_tile():
    """29 Q tiles in groups of ten: 70 positions on an XCD, two or three of them empty, keep their places in a round of 64."""
    assert _lib.attention_split_plan(0, 3, 3712, 3712, 6, 64, False)[0] in (0, 48)
    assert _lib.attention_split_plan(0, 3, 3712, 3715, 6, 64, False)[0] == 48


def test_plan_counts_the_way_of_the_parts_through_memory():
    plan = lambda *a: _lib.attention_split_plan(0, *a)
    for B, Sq, Skv, H, D in ((2, 3526, 3526, 4, 128), (8, 605, 4070, 6, 128), (2, 4352, 4608, 3, 128), (2, 3840, 3520, 4, 64),
                             (6, 2688, 2688, 5, 128), (2, 3712, 3648, 4, 64), (6, 376, 3464, 12, 128)):
        assert plan(B, Sq, Skv, H, D, False) == (0, 1)          # two or three ways: as much again as the walks save
    for B, Sq, Skv, H, D, ways in ((2, 9000, 9000, 1, 128, 3), (4, 800, 6000, 5, 128, 3), (2, 4000, 8000, 2, 64, 4)):
        assert plan(B, Sq, Skv, H, D, False)[1] >= ways


CASES = [
    # B, Sq, Skv, H, Hkv, D, causal
    (2, 300, 3500, 2, 1, 128, False),
    (2, 3600, 3600, 2, 2, 64, True),
    (3, 129, 3500, 5, 1, 32, False),
    (2, 70, 3470, 6, 3, 96, False),
    (2, 1500, 3537, 3, 3, 40, True),
    (2, 8321, 2600, 4, 2, 64, False),       # a whole round, then 16 Q tiles more
    (2, 2700, 3537, 3, 3, 40, True),        # fewer causal queries than keys
    (3, 3712, 3715, 6, 6, 64, False),       # groups of Q tiles that do not divide the sequence
]


@pytest.mark.parametrize("case", CASES)
def test_the_cases_below_are_split(case):
    B, Sq, Skv, H, Hkv, D, causal = case
    assert _lib.attention_split_plan(0, B, Sq, Skv, H, D, causal)[1] > 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, dtype):
    B, Sq, Skv, H, Hkv, D, causal = case
    q, k, v = rand((B, Sq, H, D), dtype, 1), rand((B, Skv, Hkv, D), dtype, 2), rand((B, Skv, Hkv, D), dtype, 3)
    assert _lib.attention_split_plan(q.device.index, B, Sq, Skv, H, D, causal)[1] > 1
    with torch.no_grad():
        out, lse = natten_amd.attention(q, k, v, is_causal=causal, return_lse=True)
    ref_o, ref_l = O.attention_forward(to_np(q), to_np(k), to_np(v), is_causal=causal)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("positions,splits", [(8, 2), (16, 16), (48, 5)])
def test_any_number_of_positions(positions, splits, D):
    # 48 positions of which 45 hold a Q tile; rows of the others are never written and never read
    q, k, v = rand((3, 600, 3, D), torch.bfloat16, 1), rand((3, 200, 3, D), torch.bfloat16, 2), rand((3, 200, 3, D), torch.bfloat16, 3)
    out, lse = torch.full_like(q, float("nan")), torch.full(q.shape[:-1], float("nan"), device="cuda")
    parts = torch.full((positions * splits * 128 * (D + 1),), float("nan"), device="cuda")
    L = _lib.lib()
    args = lambda p, n, pos: (q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(), p.data_ptr(), n, pos, splits,
                              _lib.DTYPE_CODES[q.dtype], 3, 600, 200, 3, 3, D, 1, D**-0.5, None, None, None,
                              torch.cuda.current_stream().cuda_stream)
    assert L.natten_amd_attention_forward_split(*args(parts, parts.numel(), positions)) == 0, L.natten_amd_last_error()
    ref_o, ref_l = O.attention_forward(to_np(q), to_np(k), to_np(v), is_causal=True)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)
    for p, n, pos in ((parts, parts.numel() - 1, positions), (parts[1:], parts.numel(), positions), (parts, 1 << 40, positions + 1),
                      (parts, 1 << 40, 512)):
        assert L.natten_amd_attention_forward_split(*args(p, n, pos)) != 0


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 96, 128])
def test_infinite_values(D):
    """Causal Q tiles with fewer key tiles than splits: a split without keys adds nothing, also where the tile that it walks
    instead holds infinities.  By rows, as in the unsplit launch (batch 1)."""
    q, k, v = (rand((2, 3600, 2, D), torch.bfloat16, seed) for seed in (1, 2, 3))
    assert _lib.attention_split_plan(q.device.index, 2, 3600, 3600, 2, D, True)[1] > 3  # more than the first Q tile has key tiles
    v[:, 5, :, 3], v[:, 40, :, 7], v[:, 3000, :, 9] = float("inf"), -float("inf"), float("inf")
    with torch.no_grad():
        out, lse = natten_amd.attention(q, k, v, is_causal=True, return_lse=True)
        alone = [natten_amd.attention(q[i : i + 1], k[i : i + 1], v[i : i + 1], is_causal=True, return_lse=True) for i in range(2)]
    want, want_lse = (torch.cat(t) for t in zip(*alone))
    assert torch.isinf(want[:, 64:, :, 3]).all() and torch.isfinite(want[..., 0]).all()
    torch.testing.assert_close(out.float(), want.float(), atol=2.0**-7, rtol=2.0**-7, equal_nan=True)  # (infinities and NaN: where they are)
    torch.testing.assert_close(lse, want_lse, atol=1e-5, rtol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("D", [64, 96, 128])
def test_rows_of_nan(D):
    """A key or a query of NaN: the rows that it reaches are NaN with an LSE of -inf, as in the unsplit launch (batch 1)."""
    q, k, v = (rand((2, 3600, 2, D), torch.bfloat16, seed) for seed in (1, 2, 3))
    q[1, 77], k[0, 3000, 1] = float("nan"), float("nan")
    with torch.no_grad():
        out, lse = natten_amd.attention(q, k, v, return_lse=True)
        alone = [natten_amd.attention(q[i : i + 1], k[i : i + 1], v[i : i + 1], return_lse=True) for i in range(2)]
    want, want_lse = (torch.cat(t) for t in zip(*alone))
    assert _lib.attention_split_plan(q.device.index, 2, 3600, 3600, 2, D, False)[1] > 1
    assert torch.isnan(want[0, :, 1]).all() and torch.isnan(want[1, 77]).all() and torch.isfinite(want[0, :, 0]).all()
    torch.testing.assert_close(out.float(), want.float(), atol=2.0**-7, rtol=2.0**-7, equal_nan=True)
    torch.testing.assert_close(lse, want_lse, atol=1e-5, rtol=1e-5)


@pytest.mark.gpu
def test_causal_queries_fewer_than_keys(monkeypatch):
    """Causal rows meet the keys up to their own number: the plan is asked for those."""
    asked, plan = [], _lib.attention_split_plan
    monkeypatch.setattr(_lib, "attention_split_plan", lambda *a: asked.append(a) or plan(*a))
    with torch.no_grad():
        for Sq, causal, split in ((1100, True, False), (512, True, False), (1100, False, True)):
            q, kv = rand((4, Sq, 2, 96), torch.bfloat16, 1), rand((4, 5568, 2, 96), torch.bfloat16, 2)
            natten_amd.attention(q, kv, kv, is_causal=causal)
            assert [a[3] for a in asked] == [Sq if causal else 5568]
            assert (plan(*asked.pop())[1] > 1) == split
