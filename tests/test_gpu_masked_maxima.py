"""GPU: the instances that take a tile's maxima from its masked logits, on walks of more tiles than are described at once;
keys of minus infinity in rows between the native head dims, whose tiles hold places past the row."""

import pytest
import torch

from natten_amd.fna import amd_fna_generic
from tests.gpu_utils import assert_close, make_qkv, oracle_full, sampled_check, to_np

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


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("shape,kernel,stride", [((40, 33), (7, 9), (1, 1)), ((9, 20, 22), (3, 5, 7), (1, 1, 2)), ((48, 48), (24, 24), (8, 8))])
def test_mostly_masked_launches_give_the_bits_of_the_work_queue(shape, kernel, stride, head_dim):
    q, k, v = make_qkv(2, shape, 4, 2, head_dim, torch.float16, seed=9)
    ones = (1,) * len(shape)
    with torch.no_grad():
        per_tile, queue = (amd_fna_generic(q, k, v, kernel, stride, ones, (False,) * len(shape), return_lse=True,
                                           run_persistent_kernel=kind, kv_splits=1) for kind in (False, True))
    assert all(torch.equal(a, b) for a, b in zip(per_tile, queue))
    sampled_check(q, k, v, *per_tile, kernel, stride, ones, (False,) * len(shape), 300, seed=1)


@pytest.mark.parametrize("head_dim", [40, 64, 72, 96, 120])
def test_keys_of_minus_infinity(head_dim):
    q, k, v = make_qkv(1, (24, 29), 2, 2, head_dim, torch.float16, seed=5)
    q[..., -1].abs_().add_(0.5)
    k[:, ::3, 1::4, :, -1] = -float("inf")  # no weight, as by a mask
    with torch.no_grad():
        out, lse = amd_fna_generic(q, k, v, (7, 9), (1, 1), (1, 1), (False, False), return_lse=True)
    ref_o, ref_l = oracle_full(q, k, v, (7, 9), (1, 1), (1, 1), (False, False))
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)
