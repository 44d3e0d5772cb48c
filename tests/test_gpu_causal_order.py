"""A causal launch of more than one round of workgroups runs the short tiles of every (batch, KV head) behind the others: which
workgroup takes which tile changes no bit, over units that do not fill the XCDs, groups of heads and counts of tiles that four
does not divide."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import bits, max_abs, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,h,hkv,d,lens", [
    (41, 390, 5, 5, 64, True), (17, 1153, 6, 2, 64, False), (30, 513, 9, 3, 128, True), (11, 1030, 6, 6, 128, False),
    (3, 9000, 4, 1, 32, True)])
def test_the_order_of_tiles_changes_no_bit(device, b, t, h, hkv, d, lens):
    g = torch.Generator(device=device).manual_seed(t)
    q, k, v = (torch.randn(b, t, n, d, generator=g, device=device).bfloat16() for n in (h, hkv, hkv))
    counts = torch.randint(1, t + 1, (b,), generator=g, device=device, dtype=torch.int32)
    keys = lambda at: KeyMask.lens(counts[at]) if lens else KeyMask.none()
    whole = svod_amd.attention(q, k, v, Attn(causal=True, keys=keys(slice(None))))
    for i in range(b):  # a row by itself is one round
        at = slice(i, i + 1)
        row = svod_amd.attention(q[at], k[at], v[at], Attn(causal=True, keys=keys(at), splits=1))
        assert (bits(whole[at]) == bits(row)).all(), i
    some = slice(0, min(t, 300))  # queries from the front see keys from the front
    p = oracle.AttnProblem(*(to_np(x[-1:, some]) for x in (q, k, v)), causal=True,
                           key_lens=np.minimum(counts[-1:].cpu().numpy(), 300) if lens else None)
    assert max_abs(to_np(whole[-1:, some]), oracle.attention_direct(p)) < 2e-2
