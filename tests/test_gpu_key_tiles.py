"""Key tiles of the dk / dv launch that begin before the first key: what the choice saves (CPU, by brute force), and the
gradients with partial first and last tiles against the CPU oracle."""

import random
from collections import Counter

import pytest
import torch

from natten_amd import _lib
from natten_amd.fna import backward_route
from natten_amd.functional import na1d, na2d, na3d
from natten_amd.tile_config import _dim_cost, _half_tile, _key_tile_dim_cost, choose_backward_role_tile_shapes
from oracle import c_oracle
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np

NA = {1: na1d, 2: na2d, 3: na3d}


def met(L, k, s, causal, tile, sub, shift):
    """Query tiles that the key tiles meet, summed, from the windows one by one, and those that need a mask."""
    pairs = Counter()
    for i in range(L):
        st = int(O.window_start(i, k, s, L, causal))
        for j in range(st, int(O.window_end(i, st, k, L, causal))):
            pairs[(j + shift) // tile, i // sub] += 1
    keys = lambda t: min((t + 1) * tile - shift, L) - max(t * tile - shift, 0)  # (no more than there are need a mask)
    return len(pairs), sum(n < keys(t) * sub for (t, _), n in pairs.items())


RULE = [(128, 32, 16), (100, 32, 16), (96, 24, 8), (90, 20, 4), (131, 33, 16), (64, 64, 16), (77, 9, 1), (200, 48, 32)]
RULE_TILES = [(8, 8), (16, 8), (32, 16), (16, 16), (128, 64), (1, 1)]


@pytest.mark.parametrize("causal", [False, True])
def test_the_choice_meets_fewer_query_tiles(causal):
    moved = 0
    for L, k, s in RULE:
        for tile, sub in RULE_TILES:
            shift = _lib.key_tile_shift(L, k, s, causal, tile, sub)
            assert 0 <= shift < tile
            if shift:
                moved += 1
                (tiles, masked), (plain, plain_masked) = (met(L, k, s, causal, tile, sub, x) for x in (shift, 0))
                assert tiles <= plain, (L, k, s, tile, sub, shift)
                # tiles and masked tiles are weighed together
                assert tiles + 0.3 * masked <= 0.95 * (plain + 0.3 * plain_masked) + 1e-9, (L, k, s, tile, sub, shift)
            assert s > 1 or shift == 0
    assert moved >= 2


def test_tile_shapes_are_chosen_for_the_tiles_as_they_lie():
    """The cost behind the tile shapes is that of the shift that the library takes."""
    rng = random.Random(4)
    problems = [(*p, c, *t) for p in RULE for c in (False, True) for t in RULE_TILES]
    for _ in range(1500):
        L = rng.choice((rng.randint(8, 200), rng.randint(200, 2500)))
        k = rng.randint(2, min(L, 200))
        problems.append((L, k, rng.randint(1, k), rng.random() < 0.4, rng.choice((2, 4, 8, 16, 32, 64, 128)), rng.choice((1, 2, 4, 8, 16, 32, 64))))
    moved = 0
    for L, k, s, causal, tile, sub in problems:
        shift = _lib.key_tile_shift(L, k, s, causal, tile, sub) if L >= tile else 0
        moved += shift > 0
        assert L < tile or _key_tile_dim_cost(L, k, s, causal, sub, tile) == _dim_cost(L, k, s, causal, sub, tile, False, shift)
    assert moved > 50


CASES = [
    # shape, kernel, stride, dilation, causal, H, Hkv, D
    ((64, 96), (32, 32), (16, 16), (1, 1), (False, False), 2, 2, 128),
    ((64, 96), (32, 32), (16, 16), (1, 1), (False, False), 4, 2, 64),
    ((50, 100), (20, 33), (4, 16), (1, 1), (False, False), 2, 1, 32),
    ((75, 68), (24, 32), (16, 16), (1, 2), (True, False), 2, 2, 64),
    ((300,), (96,), (64,), (1,), (False,), 2, 2, 128),
    ((515,), (160,), (64,), (2,), (False,), 2, 1, 32),
    ((9, 36, 40), (3, 16, 32), (1, 8, 16), (1, 1, 1), (True, False, False), 2, 2, 128),
]


def shifts_of(shape, kernel, stride, dilation, causal):
    q_tile, kv_tile = choose_backward_role_tile_shapes(shape, kernel, stride, dilation, causal)[1]
    return [_lib.key_tile_shift(-(-x // d), k, s, c, t, h)
            for x, k, s, d, c, t, h in zip(shape, kernel, stride, dilation, causal, kv_tile, _half_tile(q_tile))]


@pytest.mark.parametrize("case", CASES)
def test_the_cases_below_move_their_key_tiles(case):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    assert any(shifts_of(shape, kernel, stride, dilation, causal))
    assert backward_route(shape, kernel, stride, dilation, causal, H * D * 2, (1,), (1,))[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, dtype):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    gen = torch.Generator().manual_seed(17)
    q, d_out = (torch.randn((2, *shape, H, D), generator=gen).to(dtype).cuda() for _ in range(2))
    k, v = (torch.randn((2, *shape, Hkv, D), generator=gen).to(dtype).cuda() for _ in range(2))
    q, k, v = (t.requires_grad_(True) for t in (q, k, v))
    out = NA[len(shape)](q, k, v, kernel, stride, dilation, causal)
    grads = torch.autograd.grad(out, (q, k, v), d_out)
    refs = c_oracle.na_backward(to_np(q), to_np(k), to_np(v), to_np(d_out), kernel, stride, dilation, causal)
    tol = {torch.float16: 1e-2, torch.bfloat16: 2e-2}[dtype]  # as tests/test_gpu_backward.py
    for name, g, r in zip(("dq", "dk", "dv"), grads, refs):
        assert_close(name, to_np(g), r, atol=tol, rtol=tol)
    again = torch.autograd.grad(NA[len(shape)](q, k, v, kernel, stride, dilation, causal), (q, k, v), d_out)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))
