"""Head dims between the native ones on the tensors as they are: the bits of the same problem with rows
padded by zeros to the next native head dim."""

import pytest
import torch

from natten_amd import _lib, torch_ops
from natten_amd.fna import amd_fna_generic
from natten_amd.functional import attention, na2d
from tests.gpu_utils import assert_close, oracle_full, to_np

pytestmark = pytest.mark.gpu


def make(B, shape, H, Hkv, D, dtype, seed=0):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn((B, *shape, h, D), generator=gen).to(dtype).cuda() for h in (H, Hkv, Hkv)]


def padded(t):
    d = t.shape[-1]
    return torch.nn.functional.pad(t, (0, (64 if d < 64 else 128) - d))


CASES = [
    # shape, kernel, stride, dilation, causal
    ((16, 32), (7, 9), (1, 1), (1, 1), (False, False)),      # whole tiles
    ((19, 27), (5, 8), (2, 3), (1, 2), (False, True)),       # tiles past the group's end
    ((5, 50), (3, 17), (1, 4), (1, 1), (True, False)),       # groups narrower than a KV tile
    ((300,), (65,), (16,), (2,), (True,)),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("D", [40, 56, 72, 96, 104, 120])
def test_neighborhood(case, D):
    shape, kernel, stride, dilation, causal = case
    q, k, v = make(2, shape, 4, 2, D, torch.bfloat16 if D % 16 else torch.float16)
    args = (kernel, stride, dilation, causal, D**-0.5)
    out, lse = amd_fna_generic(q, k, v, *args, return_lse=True)
    ref, ref_lse = amd_fna_generic(padded(q), padded(k), padded(v), *args, return_lse=True, kv_splits=1)
    assert out.shape == q.shape and torch.equal(out, ref[..., :D]) and torch.equal(lse, ref_lse)
    ref_o, ref_l = oracle_full(q, k, v, kernel, stride, dilation, causal)
    assert_close("out", to_np(out), ref_o)
    assert_close("lse", to_np(lse), ref_l)


@pytest.mark.parametrize("D,S,Skv,causal", [(48, 128, 64, False), (72, 129, 77, False), (96, 1, 1, False), (96, 200, 200, True),
                                            (112, 65, 513, False)])
def test_dense(D, S, Skv, causal):
    q, _, _ = make(2, (S,), 4, 2, D, torch.bfloat16)
    _, k, v = make(2, (Skv,), 4, 2, D, torch.bfloat16, seed=1)
    out, lse = attention(q, k, v, is_causal=causal, return_lse=True)
    ref, ref_lse = attention(padded(q), padded(k), padded(v), is_causal=causal, scale=D**-0.5, return_lse=True)
    assert torch.equal(out, ref[..., :D]) and torch.equal(lse, ref_lse)


def test_no_padded_copies_and_no_neighbouring_rows(monkeypatch):
    q, k, v = make(1, (16, 16), 4, 4, 72, torch.bfloat16)
    ref = na2d(q, k, v, 5)
    monkeypatch.setattr(torch.nn.functional, "pad", None)
    # what lies behind a row in memory (the next head's) takes no part, whatever it holds
    for t in (q, k, v):
        t[..., 1::2, :] = float("nan")
    out = na2d(q, k, v, 5)
    assert torch.equal(out[..., ::2, :], ref[..., ::2, :]) and out[..., 1::2, :].isnan().all()


def test_operands_that_are_not_sixteen_byte_aligned():
    q, k, v = make(1, (16, 16), 2, 2, 96, torch.bfloat16)
    off = [torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape) for t in (q, k, v)]
    assert any(t.data_ptr() % 16 for t in off)
    assert torch.equal(na2d(*off, 5), na2d(q, k, v, 5))
    assert torch.equal(attention(*(t.flatten(1, 2) for t in off)), attention(*(t.flatten(1, 2) for t in (q, k, v))))


def test_launches_without_a_narrow_form_take_padded_copies():
    q, k, v = make(1, (32, 32), 2, 2, 96, torch.bfloat16)
    a = (7, 1, 1, False)
    ref = amd_fna_generic(q, k, v, *a)
    for kw in ({"run_persistent_kernel": True}, {"kv_splits": 2}, {"q_tile_shape": (8, 8), "kv_tile_shape": (8, 8)}, {"fused": False}):
        assert_close(str(kw), to_np(amd_fna_generic(q, k, v, *a, **kw)), to_np(ref))
    with pytest.raises(RuntimeError):  # the library refuses them
        _lib.fna_forward_fused(q, k, v, (7, 7), (1, 1), (1, 1), (False, False), 0.1, (8, 16), (8, 8), run_persistent=True)
    with pytest.raises(RuntimeError):
        torch_ops.fna_forward(q.flatten(1, 2), k.flatten(1, 2), v.flatten(1, 2), (7, 7), (1, 1), (1, 1), (False, False), 0.1,
                              (32, 32), (32, 32), (32, 32), (8, 16), (8, 8))


@pytest.mark.parametrize("D", [40, 96, 120])
def test_few_heads_share_the_key_tiles_of_a_query_tile(D):
    # 16 query tiles of 26 key tiles: left open, the call splits the key tiles as it does at native head dims
    q, k, v = make(1, (2048,), 1, 1, D, torch.bfloat16)
    args = ((1500,), (1,), (1,), (False,), D**-0.5)
    out, lse = amd_fna_generic(q, k, v, *args, return_lse=True)
    ref, ref_lse = amd_fna_generic(padded(q), padded(k), padded(v), *args, return_lse=True, kv_splits=4)
    assert torch.equal(out, ref[..., :D]) and torch.equal(lse, ref_lse)
    one, _ = amd_fna_generic(q, k, v, *args, return_lse=True, kv_splits=1)
    assert not torch.equal(out, one)
    assert_close("split against unsplit", to_np(out), to_np(one))


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("D", [56, 72, 104])
def test_split_rows_as_they_are(case, D):
    shape, kernel, stride, dilation, causal = case
    q, k, v = make(2, shape, 4, 2, D, torch.float16)
    args = (kernel, stride, dilation, causal, D**-0.5)
    out, lse = amd_fna_generic(q, k, v, *args, return_lse=True, kv_splits=3)
    ref, ref_lse = amd_fna_generic(padded(q), padded(k), padded(v), *args, return_lse=True, kv_splits=3)
    assert torch.equal(out, ref[..., :D]) and torch.equal(lse, ref_lse)
