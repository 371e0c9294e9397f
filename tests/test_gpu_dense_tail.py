"""Dense attention over key sequences that no KV tile divides: the last tile is moved back to end with the
sequence (from 64 keys on), shorter sequences are clamped; against the CPU oracle."""

import pytest
import torch

import natten_amd
from oracle import na_oracle as O
from tests.gpu_utils import assert_close, to_np
from tests.test_gpu_attention import _rand

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("D", [32, 64, 96, 128])
@pytest.mark.parametrize("Skv", [63, 64, 65, 100, 127, 129, 193])
def test_last_tile(Skv, D, causal):
    for Sq in (1, 130, Skv):
        q, k, v = _rand((2, Sq, 4, D), torch.bfloat16, Sq), _rand((2, Skv, 2, D), torch.bfloat16, 1), _rand((2, Skv, 2, D), torch.bfloat16, 2)
        with torch.no_grad():
            out, lse = natten_amd.attention(q, k, v, is_causal=causal, return_lse=True)
        ref_o, ref_l = O.attention_forward(to_np(q), to_np(k), to_np(v), is_causal=causal)
        assert_close(f"out {Sq}", to_np(out), ref_o)
        assert_close(f"lse {Sq}", to_np(lse), ref_l)
