"""Dense and packed backward whose dq launch runs beside the dk / dv launch: the bits of one behind the other, on several
streams and threads and where memory is reused at once; a captured call makes its launches one behind the other.  Where it is done
(CPU).  The two bits of the C interface's q_scaled_filled."""

import threading
import time

import pytest
import torch

from natten_amd import _lib


def test_rule():
    rule = _lib._backward_launches_overlap
    assert rule(128, 264, 128, True, False)       # packed, sequences up to 2048, four query heads a key head
    assert rule(128, 284, 282, False, True)       # a second round of 28 key tiles
    assert not rule(128, 256, 64, False, True)    # one full round
    assert not rule(128, 512, 128, False, True)
    assert not rule(128, 1440, 60, False, True)   # a last round of 160 of six
    assert not rule(128, 24, 5, False, True)      # over before a second stream has begun
    assert not rule(64, 264, 128, True, False)
    assert not rule(128, 456, 228, True, True)    # idle for a ninth of the time
    assert not rule(128, 180, 178, False, True) and not rule(128, 180, 178, False, False)  # without a mask: for three tenths


def test_rule_counts_the_compute_units_of_the_device():
    rule = _lib._backward_launches_overlap
    assert rule(128, 264, 128, True, False, 256) and not rule(128, 264, 128, True, False, 132)   # full with half of them
    assert not rule(128, 256, 128, False, True, 256) and rule(128, 256, 128, False, True, 512)    # a round that is half full


def problem(packed, seed, H=8, Hkv=2, D=128):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    B, S = (1, 1300) if packed else (2, 600)
    q, out, d_out, k, v = rand(B, S, H, D), rand(B, S, H, D), rand(B, S, H, D), rand(B, S, Hkv, D), rand(B, S, Hkv, D)
    lse = torch.rand((B, S, H), generator=gen, device="cuda") + 7
    if not packed:
        return lambda: _lib.attention_backward(q, k, v, out, d_out, lse, True, 0.088)
    cu = torch.tensor([0, 700, 701, 1100, 1290], dtype=torch.int32, device="cuda")
    return lambda: _lib.attention_backward_varlen(q, k, v, out, d_out, lse, cu, cu, True, 0.088, 700)


def test_rule_leaves_out_what_the_host_takes_longer_for():
    """Steps whose launches are over before the host has made them gain nothing from a second stream."""
    def dense(B, S, H, Hkv, causal):
        return _lib._backward_launches_overlap(128, B * -(-S // 128) * Hkv, -(-S // 64) * (H // Hkv), causal, True, 256, -(-S // 64))

    assert not dense(2, 944, 2, 1, False) and not dense(1, 1893, 16, 8, True) and not dense(2, 235, 16, 1, False)
    assert not dense(2, 2157, 8, 4, True) and not dense(1, 1418, 4, 1, True) and not dense(1, 1497, 4, 1, False)
    assert dense(1, 1710, 8, 2, False) and dense(1, 4000, 4, 4, True) and dense(2, 2552, 16, 1, True)


@pytest.mark.gpu
def test_the_device_is_asked(monkeypatch):
    units = torch.cuda.get_device_properties(0).multi_processor_count
    for packed in (False, True):
        call, asked = problem(packed, 1), []
        monkeypatch.setattr(_lib, "_backward_launches_overlap", lambda *a: asked.append(a[5]))
        call()
        assert asked == [units]


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_other_head_dims_do_not_ask(monkeypatch, packed):
    """Only head dim 128 has the two streams: a short step of another one waits for the host and does not pay for the question."""
    def asked(*a):
        raise AssertionError("asked")

    call = problem(packed, 1, D=64)
    monkeypatch.setattr(_lib, "_backward_launches_overlap", asked)
    monkeypatch.setattr(_lib, "_compute_units", asked)
    call()


@pytest.mark.gpu
def test_a_bound_of_all_rows_says_nothing(monkeypatch):
    """max_seqlen_Q as large as the batch, with several sequences in it, is no estimate of the longest."""
    asked = []
    monkeypatch.setattr(_lib, "_backward_launches_overlap", lambda *a: asked.append(a) or False)
    q, out, d_out = (torch.randn((1, 640, 4, 128), device="cuda", dtype=torch.bfloat16) for _ in range(3))
    k, v, lse = (*(torch.randn((1, 640, 2, 128), device="cuda", dtype=torch.bfloat16) for _ in range(2)), torch.rand((1, 640, 4), device="cuda"))
    for lengths, bound, asks in (((300, 340), 340, 1), ((300, 340), 640, 0), ((300, 340), 0, 0), ((640,), 640, 1)):
        cu = torch.tensor([0, *torch.tensor(lengths).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
        asked.clear()
        _lib.attention_backward_varlen(q, k, v, out, d_out, lse, cu, cu, True, 0.088, bound)
        assert len(asked) == asks, (lengths, bound)


def both_ways(monkeypatch, call):
    monkeypatch.setattr(_lib, "_backward_launches_overlap", lambda *a: False)
    serial = call()
    torch.cuda.synchronize()
    monkeypatch.setattr(_lib, "_backward_launches_overlap", lambda *a: True)
    return serial


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_same_bits(monkeypatch, packed):
    call = problem(packed, 1)
    serial = both_ways(monkeypatch, call)
    for _ in range(5):  # (the workspace of one call is memory of the next)
        copies = [t * 1 for t in call()]  # read on the caller's stream at once
        for got, want in zip(copies, serial):
            assert torch.equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_streams_and_threads(monkeypatch, packed):
    calls = [problem(packed, s) for s in (1, 2)]
    serial = [both_ways(monkeypatch, c) for c in calls]
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        for stream in (torch.cuda.Stream(), torch.cuda.Stream()):
            with torch.cuda.stream(stream):
                for _ in range(3):
                    got = [t * 1 for t in calls[i]()]
                    if not all(torch.equal(a, b) for a, b in zip(got, serial[i])):
                        wrong.append(i)
            stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_streams_of_a_thread_do_not_wait_for_each_other(monkeypatch, packed):
    """A call on one stream ends while the call before it, on another stream of the thread, still waits for its turn."""
    calls = [problem(packed, s) for s in (1, 2)]
    serial = [both_ways(monkeypatch, c) for c in calls]
    torch.cuda.synchronize()
    busy = torch.cuda.Stream()
    done = torch.cuda.Event()
    with torch.cuda.stream(busy):
        torch.cuda._sleep(10**9)  # (half a second: a spin that ends by itself)
        first = calls[0]()
        done.record()
    free = None
    for _ in range(3):  # streams share a few hardware queues: one whose own work is not behind the spin
        other = torch.cuda.Stream()
        with torch.cuda.stream(other):
            torch.zeros(1, device="cuda")
        for _ in range(200):
            if other.query():
                break
            time.sleep(1e-4)
        if other.query() and not done.query():
            free = other
            break
    if free is None:
        busy.synchronize()
        pytest.skip("no stream with a hardware queue of its own")
    with torch.cuda.stream(free):
        second = calls[1]()
    free.synchronize()
    waited = done.query()
    busy.synchronize()
    assert not waited, "the second call waited for the first one's stream"
    for got, want in zip((first, second), serial):
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True])
def test_captured(monkeypatch, packed):
    call = problem(packed, 1)
    serial = both_ways(monkeypatch, call)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call()
    for _ in range(3):
        for t in got:
            t.zero_()
        eager = call()  # (the side stream, between replays)
        graph.replay()
        torch.cuda.synchronize()
        for a, b, want in zip(got, eager, serial):
            assert torch.equal(a, want) and torch.equal(b, want)


@pytest.mark.gpu
@pytest.mark.parametrize("filled", [1, 2, 3])
@pytest.mark.parametrize("packed", [False, True])
def test_workspace_filled_or_not(packed, filled):
    """q_scaled_filled: bit 0 says whether the workspace holds the scaled queries, bit 1 asks for the second stream."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *shape: torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16)
    S, H, Hkv, D = 400, 4, 2, 128
    q, out, d_out, k, v = rand(1, S, H, D), rand(1, S, H, D), rand(1, S, H, D), rand(1, S, Hkv, D), rand(1, S, Hkv, D)
    lse = torch.rand((1, S, H), generator=gen, device="cuda") + 6
    cu = torch.tensor([0, 250, 251, 400], dtype=torch.int32, device="cuda")
    tiles = torch.empty((2, cu.numel() + 1, 2), dtype=torch.int32, device="cuda")
    scaled = torch.empty_like(q)
    neg_delta, neg_lse2 = _lib.backward_prepare(q, out, d_out, lse, D**-0.5, scaled, (cu, cu, S, tiles))

    def grads(filled):
        q_scaled = scaled if filled & 1 else torch.full_like(q, float("nan"))
        got = [torch.full_like(t, float("nan")) for t in (q, k, v)]
        head = (q.data_ptr(), k.data_ptr(), v.data_ptr(), d_out.data_ptr(), neg_lse2.data_ptr(), neg_delta.data_ptr(),
                *(g.data_ptr() for g in got), q_scaled.data_ptr(), filled, _lib.DTYPE_CODES[q.dtype])
        tail = (H, Hkv, D, 1, D**-0.5, torch.cuda.current_stream().cuda_stream)
        if packed:
            rc = _lib.lib().natten_amd_attention_backward_varlen(*head, cu.numel() - 1, S, S, cu.data_ptr(), cu.data_ptr(), tiles.data_ptr(), *tail)
        else:
            rc = _lib.lib().natten_amd_attention_backward(*head, 1, S, S, *tail)
        assert rc == 0, _lib.lib().natten_amd_last_error()
        return got

    for got, want in zip(grads(filled), grads(0)):
        assert torch.isfinite(want).all() and torch.equal(got, want)
