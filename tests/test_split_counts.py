"""The splits that a call takes which names none, at calls whose counts were timed on an MI355X: the microseconds of the counts
beside the one taken stand with each.  No device: the workspace that the rule asks for tells the count."""
import pytest
import torch

import svod_amd
from svod_amd import Attn, Cache


def t(shape):
    return torch.empty(shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("b,tq,h,hkv,d,tk,options,want", [
    # With a bias a step waits for the bias, and more of them in flight are always less time.
    (8, 96, 16, 16, 64, 3757, ("bias",), 4),       # 382.3 whole, 209.6 in two, 116.8 in four
    (5, 512, 16, 16, 64, 9083, ("bias",), 2),      # 1174.8 whole, 678.5 in two
    (12, 834, 3, 3, 128, 4911, ("bias",), 2),      # 532.7 whole, 317.0 in two
    (7, 63, 8, 4, 256, 1817, ("bias",), 3),
    # The compute unit with the most workgroups sets the pace.
    (5, 179, 16, 16, 64, 10531, (), 3),            # 95.3 in two, 71.9 in three
    (18, 131, 8, 8, 256, 7874, (), 2),             # 486.1 whole, 393.3 in two
    (3, 41, 32, 8, 128, 9405, (), 5),              # 75.1 in three, 54.7 in five
    (2, 309, 12, 12, 64, 5978, ("cache",), 7),     # 36.7 in four, 29.2 in seven
    (4, 158, 8, 8, 48, 4718, (), 8),               # 23.3 in four, 21.6 in eight
    # Full tiles whose states cost more than their steps; causal tiles see no key past their own.
    (2, 1048, 16, 2, 128, 1048, ("causal",), 1),   # 28.5 whole, 52.0 in two
    (4, 384, 16, 16, 64, 5371, ("causal",), 1),    # 11.2 whole, 20.9 in three
    (1, 3946, 8, 8, 48, 3946, ("causal",), 2),     # 47.5 whole, 37.6 in two
    (10, 512, 8, 8, 256, 1328, (), 1),             # 59.6 whole, 105.2 in two
])
def test_a_count_is_the_one_that_was_the_least_time(b, tq, h, hkv, d, tk, options, want):
    bias = t([1, h, tq, tk]) if "bias" in options else None
    cache = Cache(hkv, hkv) if "cache" in options else None
    opts = Attn(causal="causal" in options, bias=bias, cache=cache)
    got = svod_amd.ops._calls().attention_workspace(t([b, tq, h, d]), t([b, tk, 2 * hkv if cache else hkv, d]), opts)
    assert got == (0 if want == 1 else want * b * tq * h * (d + 2) * 4)
