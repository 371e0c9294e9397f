"""Rows of a sequence-packed forward that belong to no sequence: the launch that clears them against the one that leaves
them, on zeros: offsets around the 128 rows and 32 bits a workgroup looks at, gaps, offsets that are not followed, more sequences
than threads and so many that a workgroup takes more rows, sequences longer than the launch was sized for, all head dims."""

import pytest
import torch

from natten_amd import _lib

TOTAL = 700
BATCHES = {
    "every row": ([0, 31, 32, 128, 700], 572),
    "gaps at both ends": ([33, 95, 127, 129, 500], 371),
    "nothing": ([5, 5, 5], 1),
    "not followed": ([0, 40, 30, 30, 5000, 300, 699], 399),
    "longer than the launch": ([0, 400, 431, 700], 129),
    "more than threads": (list(range(0, 600, 2)), 2),
    "more rows a workgroup": ([min(i // 2, 690) for i in range(4, 5000)], 1),
}


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,heads,dtype", [(32, 3, torch.bfloat16), (64, 1, torch.float16), (128, 2, torch.bfloat16)])
@pytest.mark.parametrize("batch", BATCHES)
def test_all_rows_are_written(batch, head_dim, heads, dtype):
    offsets, longest = BATCHES[batch]
    gen = torch.Generator().manual_seed(1)
    q, k, v = (torch.randn((1, TOTAL, heads, head_dim), generator=gen).to(dtype).cuda() for _ in range(3))
    cu_q = torch.tensor(offsets, dtype=torch.int32, device="cuda")
    cu_kv = cu_q.clone()
    if batch == "every row":
        cu_kv[2] = cu_kv[1]  # a sequence without keys: zeros and -inf
    results = []
    for entry, fill in (("", 0.0), ("_all_rows", float("nan"))):
        out = torch.full_like(q, fill)
        lse = torch.full((TOTAL, heads), fill, device="cuda")
        rc = getattr(_lib.lib(), "natten_amd_attention_forward_varlen" + entry)(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), lse.data_ptr(), _lib.DTYPE_CODES[dtype], len(offsets) - 1,
            TOTAL, TOTAL, longest, longest, heads, heads, head_dim, cu_q.data_ptr(), cu_kv.data_ptr(), 1, 0.125, None, None, None,
            _lib._stream(q))
        assert rc == 0
        results.append((out, lse))
    (out0, lse0), (out1, lse1) = results
    assert torch.equal(out0, out1) and torch.equal(lse0, lse1)
