"""KV tiles are described 64 at a time and the descriptions moved on by 32: walks that end on either side of a
move, in one and several dimensions, with and without masks, whole and split; against the CPU oracle."""

import pytest
import torch

from natten_amd.fna import amd_fna_generic
from natten_amd.functional import attention
from oracle import na_oracle as O
from tests.gpu_utils import make_qkv, sampled_check, assert_close, to_np

pytestmark = pytest.mark.gpu

# shape, kernel, stride, dilation, causal, H, Hkv, D; KV tiles of a Q tile in the comment
CASES = [
    ((4160,), (3968,), (1,), (1,), (False,), 2, 1, 64),                                    # 62 .. 65
    ((4300,), (4096,), (64,), (1,), (False,), 1, 1, 128),                                  # 64 (65 with the odd start)
    ((6300,), (6000,), (1,), (1,), (True,), 1, 1, 32),                                     # 1 .. 96
    ((80, 96), (72, 80), (8, 16), (1, 1), (False, True), 2, 2, 64),                         # boxes of two dimensions
    ((9, 40, 51), (9, 33, 45), (1, 4, 1), (1, 1, 1), (False, False, False), 2, 1, 128),     # ... of three
    ((12, 46, 60), (5, 21, 27), (1, 1, 3), (2, 2, 2), (True, False, False), 2, 2, 96),
]


@pytest.mark.parametrize("splits", [None, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, dtype, splits):
    shape, kernel, stride, dilation, causal, H, Hkv, D = case
    q, k, v = make_qkv(1, shape, H, Hkv, D, dtype, seed=7)
    for launch in ([False] if splits else [False, True] if D != 96 else [False]):
        with torch.no_grad():
            out, lse = amd_fna_generic(q, k, v, kernel, stride, dilation, causal, return_lse=True, kv_splits=splits or 1,
                                       run_persistent_kernel=launch)
        sampled_check(q, k, v, out, lse, kernel, stride, dilation, causal, 300, seed=1, tag=str((splits, launch)))


@pytest.mark.parametrize("Skv", [64 * 63, 64 * 64 - 1, 64 * 64 + 1, 64 * 96, 64 * 96 + 65, 64 * 128 + 2])
def test_dense(Skv):
    gen = torch.Generator().manual_seed(Skv)
    q, k, v = (torch.randn((1, s, 2, 64), generator=gen).to(torch.bfloat16).cuda() for s in (130, Skv, Skv))
    with torch.no_grad():
        out, lse = attention(q, k, v, return_lse=True)
    ref_o, ref_l = O.attention_forward(to_np(q), to_np(k), to_np(v), is_causal=False)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)
