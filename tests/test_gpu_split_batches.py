"""The merge of key splits takes their states eight at a time: counts at and past a batch's edges."""
import numpy as np
import pytest

import oracle
import svod_amd
from svod_amd import Attn
from util import Lcg, bf16_tensor, max_abs, mean_rel, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,d,t", [(7, 64, 1), (8, 32, 1), (9, 128, 2), (16, 64, 5), (17, 48, 1), (33, 256, 1)])
def test_any_count_of_splits_merges_to_the_softmax(device, splits, d, t):
    b, h, tk = 2, 2, 64 * 33 - 5
    g = Lcg(splits)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, h, d)), g.bf16((b, tk, h, d))
    got = to_np(svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)), Attn(splits=splits)))
    assert "combine_splits" in svod_amd.chosen()
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v))
    assert max_abs(got, want) < 2e-2
    assert mean_rel(got, oracle.round_bf16(want.astype(np.float32))) < 4e-3
