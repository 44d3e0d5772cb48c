"""The causal calls that take a tile's keys in two halves at d 128: tiles over enough keys of their own, and, in a second round of
workgroups, tiles long enough for it.  The calls are ones whose two forms were timed on an MI355X, microseconds whole and in halves."""
import pytest
import torch

import svod_amd
from svod_amd import Attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,tk,h,hkv,d,sides", [
    (4, 136, 691, 16, 16, 128, False),     # 8.2, 8.9: a tile sees 136 keys
    (1, 600, 691, 4, 4, 128, True), (1, 512, 691, 4, 4, 128, False),
    (2, 142, 746, 16, 2, 128, False),      # 8.8, 9.6
    (2, 1465, 772, 16, 16, 128, False),    # 22.3, 30.4 with a mask
    (3, 1489, 1489, 8, 8, 128, True),      # 34.7, 30.5: 288 workgroups of 12 tiles a head
    (9, 1452, 1452, 4, 4, 128, False),     # 41.1, 46.6: 480
    (8, 1547, 1547, 4, 4, 128, False),     # 36.5, 43.4: 416 of 13
    (3, 1906, 1906, 8, 8, 128, True),      # 42.7, 36.1: 360 of 15
    (3, 2576, 2576, 8, 8, 128, False),     # 59.7, 67.7: 504 of 21
    (4, 2746, 2746, 4, 4, 128, True),      # 53.6, 45.1: 352 of 22
    (1, 3966, 3966, 16, 16, 128, True),    # 105.0, 80.9: 496 of 31
    (2, 2048, 2048, 16, 8, 128, True),     # 59.4, 51.9: 512 of 16, two heads over the same keys
    (5, 1500, 1500, 16, 8, 128, False), (1, 1488, 1488, 32, 8, 128, True),  # in groups 480 of 12 and 384
    (2, 137, 563, 12, 12, 64, True),       # d 64: 0.94 to 0.98 times
])
def test_causal_lines(device, b, t, tk, h, hkv, d, sides):
    q = torch.zeros(b, t, h, d, dtype=torch.bfloat16, device=device)
    k = torch.zeros(b, tk, hkv, d, dtype=torch.bfloat16, device=device)
    v = torch.ones_like(k)
    # (A lent workspace of a few bytes: the keys are not split.)
    got = svod_amd.attention(q, k, v, Attn(causal=True), workspace=torch.empty(16, dtype=torch.uint8, device=device))
    assert ("sides: 2" in svod_amd.chosen()) == sides, svod_amd.chosen()
    assert bool((got == 1.0).all())
