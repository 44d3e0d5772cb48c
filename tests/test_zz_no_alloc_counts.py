"""svodk_attention_noalloc with no count named: what svodk_attention gives for the count that fits the static array, bit for bit.  An unsplit call keeps its keys whole where svodk_attention takes a tile's keys in two halves, and a count of the rule's own is
lowered to what the array holds, to several and to one."""
import numpy as np
import pytest
import torch

import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, bits

pytestmark = pytest.mark.gpu


def operands(device, b, t, tk, h, hkv, d):
    g = Lcg(71)
    return tuple(bf16_tensor(g.bf16(s), device) for s in ((b, t, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))


@pytest.mark.parametrize("b,t,tk,h,hkv,d,causal", [(1, 1500, 1500, 16, 16, 64, False), (2, 700, 700, 8, 4, 128, True),
                                                   (3, 130, 600, 2, 2, 64, False)])
def test_an_unsplit_call_keeps_its_keys_whole(device, b, t, tk, h, hkv, d, causal):
    q, k, v = operands(device, b, t, tk, h, hkv, d)
    keys = KeyMask.lens(torch.tensor([tk - 90 * i for i in range(b)], dtype=torch.int32, device=device))
    asked = svod_amd.ops._calls().attention_workspace(q, k, Attn(causal=causal, keys=keys))
    assert asked == 0  # the rule asks for no split
    got = svod_amd.attention_noalloc(q, k, v, Attn(causal=causal, keys=keys), torch.full_like(q, float("nan")))
    whole = svod_amd.chosen()
    want = svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys, splits=1))
    assert svod_amd.chosen() == whole and "sides: 2" not in whole
    assert np.array_equal(bits(got), bits(want))
    svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys))
    assert "sides: 2" in svod_amd.chosen()


@pytest.mark.parametrize("t,want", [(256, 3), (512, 1)])
def test_the_rules_count_shrinks_to_the_array(device, t, want):
    tk, h, d = 8192, 16, 128
    q, k, v = operands(device, 1, t, tk, h, h, d)
    per_split, room = t * h * (d + 2) * 4, svod_amd.noalloc_scratch_bytes()
    asked = svod_amd.ops._calls().attention_workspace(q, k, Attn())
    assert asked > room and asked // per_split > want == room // per_split  # else this call tests nothing
    got = svod_amd.attention_noalloc(q, k, v, Attn(), torch.full_like(q, float("nan")))
    assert ("combine_splits" in svod_amd.chosen()) == (want > 1) and "sides: 2" not in svod_amd.chosen()
    assert np.array_equal(bits(got), bits(svod_amd.attention(q, k, v, Attn(splits=want))))
