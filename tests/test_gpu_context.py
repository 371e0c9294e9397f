"""Windows and context in one launch: context lengths around whole tiles, every head dim and tile pair that has the launch,
windows of one KV tile, GQA, dilation, causal dimensions, edge tiles; against the CPU oracle (two attentions merged in
float64).  Problems without such a launch still merge two."""

import numpy as np
import pytest
import torch

from natten_amd import _lib
from natten_amd.fna import _context_call_plan, amd_fna_with_context
from natten_amd.functional import attention, merge_attentions, na1d, na2d, na3d
from natten_amd.tile_config import choose_fitting_forward_tiles
from oracle import c_oracle
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np

NA = {1: na1d, 2: na2d, 3: na3d}

CASES = [
    # shape, kernel, stride, dilation, causal, H, Hkv, D
    ((40, 33), (7, 7), (1, 1), (1, 1), (False, False), 4, 2, 64),        # 64 x 64 tiles
    ((40, 33), (7, 7), (1, 2), (1, 1), (True, False), 2, 2, 32),
    ((37, 44), (8, 11), (2, 1), (2, 1), (True, False), 4, 1, 128),
    ((24, 40), (9, 17), (3, 1), (1, 1), (False, True), 2, 2, 96),
    ((24, 40), (9, 17), (3, 1), (1, 1), (False, False), 2, 1, 40),
    ((256,), (64,), (64,), (1,), (False,), 2, 2, 128),                    # one window tile, then the context
    ((700,), (130,), (1,), (3,), (False,), 2, 1, 72),
    ((9, 16, 24), (5, 8, 11), (1, 8, 2), (1, 1, 2), (True, False, False), 2, 2, 64),
    ((30, 40), (21, 21), (1, 1), (1, 1), (False, False), 2, 2, 128),      # the cheapest KV tile is wider than the input, split windows
]


def inputs(case, context, dtype):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    gen = torch.Generator().manual_seed(context)
    rand = lambda *s: torch.randn(s, generator=gen).to(dtype).cuda()
    return rand(2, *shape, H, D), rand(2, *shape, Hkv, D), rand(2, *shape, Hkv, D), rand(2, context, Hkv, D), rand(2, context, Hkv, D)


def reference(case, q, k, v, ck, cv):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    o, l = c_oracle.na_forward(to_np(q), to_np(k), to_np(v), kernel, stride, dilation, causal)
    flat = to_np(q).reshape(2, -1, H, D)
    co, cl = O.attention_forward(flat, to_np(ck), to_np(cv), is_causal=False)
    co, cl = np.asarray(co, dtype=np.float64).reshape(o.shape), np.asarray(cl, dtype=np.float64).reshape(l.shape)
    lse = np.logaddexp(l, cl)
    return np.exp(l - lse)[..., None] * o + np.exp(cl - lse)[..., None] * co, lse


@pytest.mark.parametrize("case", CASES)
def test_the_cases_below_have_the_launch(case):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    assert _context_call_plan(torch.bfloat16, (2, *shape, H, D), Hkv, kernel, stride, dilation, causal, None) is not None


@pytest.mark.parametrize("shape,kernel,dilation", [((64, 7, 1000), (8, 5, 2), (2, 1, 1)), ((64, 5, 3000), (8, 5, 2), (2, 1, 1)),
                                                   ((64, 7, 3000), (8, 3, 2), (1, 1, 1))])
def test_tiles_that_span_too_much_merge_two(shape, kernel, dilation):
    """Groups narrower than the cheapest KV tile, and the fitting one spans more than the launch addresses: no joint launch."""
    ones, causal = (1, 1, 1), (False,) * 3
    assert choose_fitting_forward_tiles(shape, kernel, ones, dilation, causal) is not None
    assert _context_call_plan(torch.bfloat16, (1, *shape, 32, 128), 32, kernel, ones, dilation, causal, None) is None
    assert _context_call_plan(torch.bfloat16, (1, *shape, 2, 128), 2, kernel, ones, dilation, causal, None) is not None


def test_long_contexts_of_padded_q_tiles_merge_two():
    """A joint walk meets the context once per Q tile of the windows: not where those are many more than dense attention's."""
    def joint(batch, shape, heads, head_dim, kernel, context):
        n = len(shape)
        return _context_call_plan(torch.bfloat16, (batch, *shape, heads, head_dim), heads, kernel, (1,) * n, (1,) * n, (False,) * n,
                                  None, context) is not None

    for D in (32, 64, 96, 128):
        for shape in ((17, 33, 9), (5, 5, 300), (13, 37, 21)):
            assert joint(2, shape, 16, D, (3, 5, 5), 128) and not joint(2, shape, 16, D, (3, 5, 5), 3072)
        assert joint(2, (10000,), 16, D, (200,), 3072) and joint(1, (30, 48, 40), 4, D, (3, 5, 5), 2048)
        assert joint(2, (64, 64), 8, D, (13, 13), 128) and joint(2, (128, 128), 16, D, (7, 9), 1024)
    assert not joint(2, (17, 33, 9), 16, 64, (3, 5, 5), 1024) and not joint(2, (64, 64), 16, 64, (7, 9), 4096)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("context", [64, 65, 77, 127, 128, 256, 4100])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, context, dtype):
    if context > 256 and case is not CASES[0] and case is not CASES[2]:
        pytest.skip("a walk past a move of the tile descriptions: one case per tile pair")
    shape, kernel, stride, dilation, causal = case[:5]
    q, k, v, ck, cv = inputs(case, context, dtype)
    with torch.no_grad():
        out, lse = NA[len(shape)](q, k, v, kernel, stride, dilation, causal, additional_keys=ck, additional_values=cv, return_lse=True)
        assert amd_fna_with_context(q, k, v, ck, cv, kernel, stride, dilation, causal, q.shape[-1] ** -0.5) is not None
    ref_o, ref_l = reference(case, q, k, v, ck, cv)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)


@pytest.mark.gpu
@pytest.mark.parametrize("case", [c for c in CASES if c[-1] in (32, 64, 128)])
def test_work_queue_gives_the_same_bits(case):
    shape, kernel, stride, dilation, causal = case[:5]
    q, k, v, ck, cv = inputs(case, 130, torch.bfloat16)
    with torch.no_grad():
        queue, plain = (NA[len(shape)](q, k, v, kernel, stride, dilation, causal, additional_keys=ck, additional_values=cv,
                                       return_lse=True, run_persistent_kernel=kind) for kind in (True, False))
    assert all(torch.equal(a, b) for a, b in zip(queue, plain))


@pytest.mark.gpu
def test_without_the_launch_two_attentions_are_merged():
    case = ((40, 33), (7, 7), (1, 1), (1, 1), (False, False), 4, 2, 64)
    shape, kernel, stride, dilation, causal = case[:5]
    for context, extra in ((63, {}), (1, {}), (128, dict(q_tile_shape=(8, 16), kv_tile_shape=(8, 8)))):
        q, k, v, ck, cv = inputs(case, context, torch.bfloat16)
        with torch.no_grad():
            out, lse = na2d(q, k, v, kernel, additional_keys=ck, additional_values=cv, return_lse=True, **extra)
            if not extra:
                assert amd_fna_with_context(q, k, v, ck, cv, kernel, stride, dilation, causal, 0.125) is None
        ref_o, ref_l = reference(case, q, k, v, ck, cv)
        assert_close("out", to_np(out), ref_o)
        assert_close("lse", to_np(lse), ref_l)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_a_result_type_that_the_caller_chooses_merges_two(dtype):
    """The joint launch rounds to the operands' type.  A float32 result is that of the merge in float32; a type that the merge
    does not take is refused."""
    case = ((40, 33), (7, 7), (1, 1), (1, 1), (False, False), 4, 2, 64)
    kernel = case[1]
    q, k, v, ck, cv = inputs(case, 128, dtype)
    v, cv = v + 3, cv + 3  # (rounding errors of one sign and size in both parts: the merge averages them)
    context = dict(additional_keys=ck, additional_values=cv, return_lse=True)
    with torch.no_grad():
        out, lse = na2d(q, k, v, kernel, out_dtype=torch.float32, **context)
        parts = na2d(q, k, v, kernel, out_dtype=torch.float32, return_lse=True), attention(
            q.flatten(1, 2), ck, cv, out_dtype=torch.float32, return_lse=True)
        want, want_lse = merge_attentions(*([t.flatten(1, 2) for t in pair] for pair in zip(*(
            (o.reshape(out.shape), l.reshape(lse.shape)) for o, l in parts))))
        assert out.dtype == torch.float32 and torch.equal(out, want.reshape(out.shape)) and torch.equal(lse, want_lse.reshape(lse.shape))
        with pytest.raises(NotImplementedError):
            na2d(q, k, v, kernel, out_dtype=torch.float64, **context)
    ref_o, _ = reference(case, q, k, v, ck, cv)
    error = lambda t: float(np.linalg.norm(to_np(t) - ref_o) / np.linalg.norm(ref_o))
    joint = amd_fna_with_context(q, k, v, ck, cv, *case[1:5], 0.125)[0]
    print(f"error of a float32 result {error(out):.3e}, of the joint launch {error(joint):.3e}")
    assert error(out) < error(joint)


@pytest.mark.gpu
def test_library_refuses_what_it_has_no_kernel_for():
    q = torch.zeros((1, 40, 33, 2, 64), dtype=torch.bfloat16, device="cuda")
    ctx = torch.zeros((1, 128, 2, 64), dtype=torch.bfloat16, device="cuda")
    args = ((7, 7), (1, 1), (1, 1), (False, False), 0.125)
    for c, tiles in ((ctx[:, :63].contiguous(), ((8, 16), (8, 8))), (ctx, ((16, 16), (8, 8)))):
        with pytest.raises(RuntimeError):
            _lib.fna_forward_fused_context(q, q, q, c, c, *args, *tiles)
