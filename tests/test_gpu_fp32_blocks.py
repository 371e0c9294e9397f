"""GPU: the float32 kernel's blocks of keys: more of them than a wave describes at once, blocks at the edges of dilation groups, and blocks
that span more than 32-bit offsets reach."""

import numpy as np
import pytest
import torch

import natten_amd
from oracle import c_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("head_dim", [8, 32, 40, 64, 128])
@pytest.mark.parametrize("layout,k,s,d,c", [
    ((45, 47), (41, 43), (1, 2), (1, 1), (False, False)),        # 126 blocks
    ((2100,), (1040,), (3,), (2,), (True,)),                      # one block more than 64
    ((9, 11, 13), (3, 5, 4), (1, 2, 1), (2, 1, 3), (False, True, False)),
    ((5,), (2,), (1,), (2,), (False,)),                           # groups of two and three keys
])
def test_blocks_against_the_oracle(layout, k, s, d, c, head_dim):
    gen = torch.Generator().manual_seed(head_dim)
    q, kk, v = (torch.randn((1, *layout, h, head_dim), generator=gen) for h in (2, 1, 1))
    out, lse = getattr(natten_amd, f"na{len(layout)}d")(q.cuda(), kk.cuda(), v.cuda(), k, s, d, c, return_lse=True)
    ref_o, ref_l = c_oracle.na_forward(q.numpy(), kk.numpy(), v.numpy(), k, s, d, c)
    assert np.abs(out.cpu().numpy() - ref_o).max() <= 1e-4 and np.abs(lse.cpu().numpy() - ref_l).max() <= 1e-4


def test_blocks_that_span_more_than_four_gigabytes():
    # sixteen keys along dimension 0, 70000 rows of 4 KB apart
    heads, head_dim, width, row = 8, 128, 70000, 16
    gen = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn((1, row, width, heads, head_dim), generator=gen, device="cuda") for _ in range(3))
    out, lse = natten_amd.na2d(q, k, v, (16, 3), return_lse=True)
    for x, y in ((0, 0), (15, 0), (3, 1), (7, 34567), (15, 69999), (0, 69998), (11, 65536)):
        first = min(max(y - 1, 0), width - 3)
        keys, values = (t[0, :, first : first + 3].reshape(-1, heads, head_dim).double() for t in (k, v))
        logits = torch.einsum("hd,nhd->hn", q[0, x, y].double(), keys) * head_dim**-0.5
        ref = torch.einsum("hn,nhd->hd", logits.softmax(-1), values)
        assert (out[0, x, y].double() - ref).abs().max() <= 1e-4
        assert (lse[0, x, y].double() - logits.logsumexp(-1)).abs().max() <= 1e-4
