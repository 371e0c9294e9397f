"""The tile walk of sequence-packed attention (backward kernels): sequence counts around the 64 that one
step of the walk takes, empty sequences, lengths around the 128-row tile, rows in front of and behind
the sequences.  Gradients against the float64 oracle at the tolerance of the backward tests (bf16 2e-2:
P and dS are rounded to bf16 before the second product)."""

import numpy as np
import pytest
import torch

import natten_amd
from natten_amd import _lib
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_seqs,head,tail", [(1, 0, 5), (63, 3, 0), (64, 0, 0), (65, 130, 257), (130, 1, 1)])
def test_every_row_is_covered_once(num_seqs, head, tail):
    rng = np.random.default_rng(num_seqs)
    lens = rng.choice([0, 1, 5, 63, 64, 127, 128, 129], size=num_seqs)
    lens[0], lens[-1] = 129, 128
    cu_list = head + np.concatenate([[0], np.cumsum(lens)])
    total = int(cu_list[-1]) + tail
    gen = torch.Generator().manual_seed(num_seqs)
    q, d_out = (torch.randn((1, total, 2, 32), generator=gen).bfloat16().cuda() for _ in range(2))
    k, v = (torch.randn((1, total, 1, 32), generator=gen).bfloat16().cuda() for _ in range(2))
    cu = torch.tensor(cu_list, dtype=torch.int32, device="cuda")
    for t in (q, k, v):
        t.requires_grad_(True)
    causal = num_seqs % 2 == 1
    out = natten_amd.attention(q, k, v, is_causal=causal, cumulative_seqlen_Q=cu, cumulative_seqlen_KV=cu, max_seqlen_Q=129,
                               max_seqlen_KV=129)
    out.backward(d_out)
    grads = [to_np(t.grad) for t in (q, k, v)]
    owned = np.zeros(total, dtype=bool)
    for a, b in zip(cu_list[:-1], cu_list[1:]):
        owned[a:b] = True
    for g in grads + [to_np(out)]:
        assert np.isfinite(g).all() and not g[:, ~owned].any()
    for i in list(range(min(num_seqs, 8))) + list(range(max(num_seqs - 8, 0), num_seqs)):
        a, b = int(cu_list[i]), int(cu_list[i + 1])
        if a == b:
            continue
        ref = O.attention_backward(*(to_np(t[:, a:b]) for t in (q, k, v, d_out)), is_causal=causal)
        for name, g, r in zip(("dq", "dk", "dv"), grads, ref):
            assert_close(f"{name} of sequence {i} of {num_seqs}, {b - a} rows", g[:, a:b], r, atol=2e-2, rtol=2e-2)


def test_time_grows_with_the_sequences_not_with_their_square():
    # 16 rows a sequence: eight times the sequences are eight times the tiles.  Finding a tile's sequence by
    # counting through all lengths in every workgroup made it 64 times the counting (52 times the time; now 6.4).
    def step(num_seqs):
        cu = torch.arange(num_seqs + 1, dtype=torch.int32, device="cuda") * 16
        q, k, v = (torch.randn((1, 16 * num_seqs, 4, 64), device="cuda", dtype=torch.bfloat16).requires_grad_(True) for _ in range(3))
        out = natten_amd.attention(q, k, v, cumulative_seqlen_Q=cu, cumulative_seqlen_KV=cu, max_seqlen_Q=16, max_seqlen_KV=16)
        d_out = torch.randn_like(out)
        best = float("inf")
        for _ in range(5):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            torch.autograd.grad(out, (q, k, v), d_out, retain_graph=True)
            end.record()
            torch.cuda.synchronize()
            best = min(best, start.elapsed_time(end))
        return best

    assert step(16384) < 16 * step(2048)


def _packed_backward(cu_q, cu_kv, rows, D):
    """Gradients of the library's packed backward for any cumulative lengths, from made-up saved tensors."""
    gen = torch.Generator().manual_seed(D)
    q, d_out, out = (torch.randn((1, rows, 2, D), generator=gen).bfloat16().cuda() for _ in range(3))
    k, v = (torch.randn((1, rows, 1, D), generator=gen).bfloat16().cuda() for _ in range(2))
    lse = (torch.randn((1, rows, 2), generator=gen) + 6).cuda()
    cus = [torch.tensor(cu, dtype=torch.int32, device="cuda") for cu in (cu_q, cu_kv)]
    return _lib.attention_backward_varlen(q, k, v, out, d_out, lse, *cus, False, D**-0.5)


@pytest.mark.parametrize("D", [32, 128])
def test_malformed_lengths_are_not_followed(D):
    # the first sequence is well-formed on both sides; the second's end lies past the rows, before them, or before its start
    ref = _packed_backward([0, 40], [0, 40], 200, D)
    for g in ref:
        assert g[:, :40].any() and not g[:, 40:].any()
    for tail in (5000, -7, 20):
        for a, b in (([0, 40, tail], [0, 40, 200]), ([0, 40, 200], [0, 40, tail])):
            for name, g, r in zip(("dq", "dk", "dv"), _packed_backward(a, b, 200, D), ref):
                assert torch.equal(g, r), (name, a, b)


@pytest.mark.parametrize("D", [32, 128])
def test_rows_behind_overlapping_sequences_are_written(D):
    # lengths that run back and forth over the same rows: the rows behind them belong to no sequence and get
    # zeros (dq doubles as the workspace of the scaled queries: a row that no tile visits would keep those)
    ref = _packed_backward([0, 1024], [0, 1024], 1300, D)
    cu = [0, 1024] * 20
    for name, g, r in zip(("dq", "dk", "dv"), _packed_backward(cu, cu, 1300, D), ref):
        assert torch.equal(g, r), name
    # one overlap on one side: the rows that only the overlapping sequence holds get zeros
    dq, dk, dv = _packed_backward([0, 60, 40, 100], [0, 50, 80, 120], 300, D)
    rq, rk, rv = _packed_backward([0, 60], [0, 50], 300, D)
    assert torch.equal(dq, rq)
    for g, r in ((dk, rk), (dv, rv)):
        assert torch.equal(g[:, :50], r[:, :50]) and not g[:, 50:80].any() and not g[:, 120:].any() and g[:, 80:120].any()
