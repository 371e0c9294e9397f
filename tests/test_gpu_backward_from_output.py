"""GPU: the backward whose dq launch comes first and prepares what the dk / dv launch reads, bit for bit against the same launches
behind natten_amd_backward_prepare; extents that no tile divides, dilation groups of two lengths, shared key / value heads."""

import pytest
import torch

import natten_amd
from natten_amd import _lib, fna
from natten_amd.tile_config import BACKWARD_TILE_SIZE, choose_tile_shapes

pytestmark = pytest.mark.gpu

CASES = [((300,), 2, 1, (31,), (4,), (1,), (True,)), ((37, 51), 4, 2, (9, 11), (2, 3), (2, 1), (False, False)),
         ((9, 17, 20), 2, 2, (3, 5, 7), (1, 1, 2), (1, 1, 2), (True, False, False)), ((16, 16), 1, 1, (5, 5), (1, 1), (1, 1), (False, False))]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [32, 64, 128])
@pytest.mark.parametrize("layout,heads,heads_kv,k,s,d,c", CASES)
def test_bits_of_the_prepared_launches(layout, heads, heads_kv, k, s, d, c, head_dim, dtype):
    gen = torch.Generator().manual_seed(head_dim)
    q, kk, v, d_out = (torch.randn((2, *layout, h, head_dim), generator=gen).to(dtype).cuda() for h in (heads, heads_kv, heads_kv, heads))
    with torch.no_grad():
        out, lse = getattr(natten_amd, f"na{len(layout)}d")(q, kk, v, k, s, d, c, return_lse=True)
    pair = choose_tile_shapes(layout, k, s, d, c, BACKWARD_TILE_SIZE, BACKWARD_TILE_SIZE)
    fused, tiles, role = fna.backward_route(layout, k, s, d, c, heads * head_dim * 2, *pair)
    if not fused:
        fused, tiles, role = fna.backward_route(layout, k, s, d, c, heads * head_dim * 2, *pair, role_tiles=False)
    if not fused:
        pytest.skip("a dilation group is narrower than every tile")
    got = _lib.fna_backward_fused(q, kk, v, d_out, lse, None, k, s, d, c, head_dim**-0.5, *tiles, *role, out=out)
    # the same launches behind the pass that prepares their arrays
    ref = tuple(torch.zeros_like(t) for t in (q, kk, v))
    scaled = torch.empty_like(q)
    neg_delta, neg_lse2 = _lib.backward_prepare(q, out, d_out, lse, head_dim**-0.5, scaled)
    L, own = _lib.lib(), role[0] is not None
    for roles, qt, kt in ((2, *(role if own else tiles)), (1, *tiles)):
        _lib._check(L.natten_amd_fna_backward_fused(
            q.data_ptr(), kk.data_ptr(), v.data_ptr(), d_out.data_ptr(), neg_lse2.data_ptr(), neg_delta.data_ptr(),
            *(t.data_ptr() for t in ref), scaled.data_ptr(), _lib.DTYPE_CODES[dtype], len(layout), 2, heads, heads_kv, head_dim,
            *_lib._problem_arrays(layout, k, s, d, c, qt, kt), head_dim**-0.5, roles + 4 + (8 if own else 0), _lib._stream(q)))
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.mark.parametrize("layout,heads,heads_kv,k,s,d,c", CASES[1:3])
def test_without_room_for_the_scaled_queries(layout, heads, heads_kv, k, s, d, c, monkeypatch):
    gen = torch.Generator().manual_seed(7)
    q, kk, v, d_out = (torch.randn((2, *layout, h, 64), generator=gen).bfloat16().cuda() for h in (heads, heads_kv, heads_kv, heads))
    q, kk, v = (t.requires_grad_(True) for t in (q, kk, v))
    out = getattr(natten_amd, f"na{len(layout)}d")(q, kk, v, k, s, d, c)
    ref = torch.autograd.grad(out, (q, kk, v), d_out, retain_graph=True)
    empty_like, of_q = torch.empty_like, []

    def full_memory(t, *args, **kwargs):
        if t.shape == q.shape:
            of_q.append(1)
        if len(of_q) == (2 if heads != heads_kv else 4):  # dq (and dk, dv of q's shape) before it
            raise torch.OutOfMemoryError("no room")
        return empty_like(t, *args, **kwargs)

    monkeypatch.setattr(torch, "empty_like", full_memory)
    got = torch.autograd.grad(out, (q, kk, v), d_out)
    assert len(of_q) == (2 if heads != heads_kv else 4)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))


def test_refusals():
    L, t = _lib.lib(), torch.zeros((1, 64, 1, 32), dtype=torch.float16, device="cuda")
    f = torch.zeros((1, 64, 1), device="cuda")
    arrays = _lib._problem_arrays((64,), (5,), (1,), (1,), (False,), (64,), (64,))

    def call(q_scaled, role):
        return L.natten_amd_fna_backward_from_output(
            *(t.data_ptr(),) * 5, f.data_ptr(), *(t.data_ptr(),) * 3, q_scaled, f.data_ptr(), f.data_ptr(), 0, 1, 1, 1, 1, 32, *arrays,
            *role, 1.0, _lib._stream(t))

    assert call(t.data_ptr(), (None, None)) != 0 and b"must not be dq" in L.natten_amd_last_error()
    other = torch.zeros_like(t)
    assert call(other.data_ptr(), (arrays[-1], None)) != 0 and b"given together" in L.natten_amd_last_error()
    assert call(other.data_ptr(), (None, None)) != 0 and b"128 tokens" in L.natten_amd_last_error()
    assert call(None, (None, None)) != 0 and b"null pointer" in L.natten_amd_last_error()
