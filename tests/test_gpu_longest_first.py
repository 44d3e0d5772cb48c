"""A call with key lengths over a few rows takes its rows longest first: every row is still computed, once, whatever the
lengths (ties, empty rows, lengths past the keys), with the bits of the call that names the order itself."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, bits, max_abs, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens,dtype,d,causal", [
    ([300, 300, 300], torch.int32, 64, False), ([0, 257, 0, 1, 999], torch.int64, 64, False),
    ([5 * i % 16 * 20 for i in range(16)], torch.int32, 64, True), ([300 - i for i in range(16)], torch.int64, 128, True),
    ([-3, 17, 300], torch.int32, 32, False), ([1 + 18 * i for i in range(17)], torch.int32, 64, False)])
def test_rows_of_any_lengths(device, lens, dtype, d, causal):
    b, t, h, hkv = len(lens), 300, 4, 2
    g = Lcg(7 + b)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, t, hkv, d)), g.bf16((b, t, hkv, d))
    dev = [bf16_tensor(x, device) for x in (q, k, v)]
    keys = KeyMask.lens(torch.tensor(lens, dtype=dtype, device=device))
    got = svod_amd.attention(*dev, Attn(causal=causal, keys=keys))
    named = torch.arange(b, dtype=torch.int32, device=device)
    assert np.array_equal(bits(got), bits(svod_amd.attention(*dev, Attn(causal=causal, keys=keys, row_order=named))))
    held = np.clip(np.asarray(lens), 0, t)
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, causal=causal, key_lens=held))
    assert max_abs(to_np(got), want) < 2e-2
