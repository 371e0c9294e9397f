"""GPU: the instances that take a tile's maxima from its masked logits, on walks of more tiles than are described at once."""

import pytest
import torch

from natten_amd.fna import amd_fna_generic
from tests.gpu_utils import make_qkv, sampled_check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("shape,kernel,stride,causal,tiles", [
    ((73, 70), (61, 59), (1, 3), (False, False), ((8, 8), (8, 8))),        # 64 .. 81 tiles of a query tile
    ((4200,), (4001,), (1,), (True,), ((64,), (64,))),                     # 1 .. 64
    ((11, 43, 45), (7, 29, 31), (1, 1, 2), (False, True, False), ((4, 4, 4), (4, 4, 4))),
])
def test_walks_of_small_tiles(shape, kernel, stride, causal, tiles, head_dim):
    q, k, v = make_qkv(1, shape, 2, 1, head_dim, torch.bfloat16, seed=head_dim)
    ones = (1,) * len(shape)
    with torch.no_grad():
        out, lse = amd_fna_generic(q, k, v, kernel, stride, ones, causal, return_lse=True, q_tile_shape=tiles[0],
                                   kv_tile_shape=tiles[1])
    sampled_check(q, k, v, out, lse, kernel, stride, ones, causal, 300, seed=1)
