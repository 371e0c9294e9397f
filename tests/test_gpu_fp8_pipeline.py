"""The 8-bit kernel forms O a tile behind the probabilities: walks of one tile to past a move of the tile descriptions,
odd and even, with row maxima that keep growing along the keys (every tile then rescales, and O an iteration late);
against the oracle at the tolerance of test_gpu_fp8."""

import pytest
import torch

import natten_amd
from oracle import c_oracle
from tests.gpu_utils import assert_close, to_np
from tests.test_gpu_fp8 import check_out, dequantise, quantise_per_head

pytestmark = pytest.mark.gpu

NA = {1: natten_amd.na1d, 2: natten_amd.na2d, 3: natten_amd.na3d}
CASES = [
    # shape, kernel, stride, causal
    ((256,), (64,), (64,), (False,)),          # one tile
    ((256,), (128,), (128,), (False,)),        # two, no mask
    ((320,), (100,), (1,), (False,)),          # three and four
    ((4224,), (4096,), (1,), (False,)),        # 64 to 67
    ((6400,), (6209,), (1,), (True,)),         # 2 to 100
    ((24, 40), (9, 17), (3, 1), (False, True)),
    ((9, 16, 24), (5, 8, 11), (1, 8, 2), (True, False, False)),
]


@pytest.mark.parametrize("ramp", [0.0, 40.0])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("case", CASES)
def test_matches_oracle(case, D, ramp):
    shape, kernel, stride, causal = case
    gen = torch.Generator().manual_seed(11)
    q, k, v = (torch.randn((1, *shape, 2, D), generator=gen).cuda() for _ in range(3))
    if ramp:
        # the logit of key i grows by `ramp` over the sequence, for every query alike
        q[..., 0] = D**0.5 / 4
        k[..., 0] = torch.linspace(0, ramp / 4, k[..., 0, 0].numel()).reshape(*shape, 1).cuda() * 4
    (q8, sq), (k8, sk), (v8, sv) = (quantise_per_head(t, torch.float8_e4m3fn) for t in (q, k, v))
    qd, kd, vd = dequantise(q8, sq), dequantise(k8, sk), dequantise(v8, sv)
    ones = (1,) * len(shape)
    for launch in (False, True):
        with torch.no_grad():
            out, lse = NA[len(shape)](q8, k8, v8, kernel, stride, ones, causal, return_lse=True, q_scale=sq, k_scale=sk,
                                      v_scale=sv, out_dtype=torch.bfloat16, run_persistent_kernel=launch)
        ref_o, ref_l = c_oracle.na_forward(to_np(qd), to_np(kd), to_np(vd), kernel, stride, ones, causal, threads=16)
        check_out(f"out {launch}", True, to_np(out), ref_o, vd)
        assert_close(f"lse {launch}", to_np(lse), ref_l)
