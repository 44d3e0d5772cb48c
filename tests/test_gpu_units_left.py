"""A launch whose (batch, KV head) pairs are no multiple of the eight XCDs shares the pairs left over out to all of them:
every query row of every head is written, with pairs fewer than XCDs, one left and seven left, one tile and several."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, max_abs, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("key_tiles")]

# (b, t, h, hkv, d, options)
CASES = [
    (1, 130, 1, 1, 64, {}),                       # one pair, two tiles: six XCDs have none
    (1, 700, 3, 3, 64, {}),                       # 18 workgroups in runs of 3
    (3, 257, 3, 3, 64, {"lens": [257, 1, 100]}),  # nine pairs: one is left
    (1, 129, 15, 15, 32, {}),                     # seven are left
    (1, 300, 10, 2, 128, {}),                     # a group's heads and tiles in one unit
    (5, 65, 3, 1, 48, {"lens": [65, 0, 64, 3, 9]}),
    (1, 300, 12, 12, 64, {"window": (64, 64)}),
    (1, 200, 12, 12, 64, {"splits": 3}),
    (1, 20, 12, 3, 64, {}),                       # grouped: a workgroup a unit
    (1, 140, 9, 3, 256, {}),
    (2, 300, 6, 3, 64, {"causal": True}),         # causal launches keep whole rounds
]


@pytest.mark.parametrize("b,t,h,hkv,d,options", CASES, ids=[f"{c[0]}x{c[1]} {c[2]}/{c[3]}x{c[4]} {' '.join(c[5])}" for c in CASES])
def test_pairs_left_over_are_computed_once_each(device, b, t, h, hkv, d, options):
    g = Lcg(17)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, t, hkv, d)), g.bf16((b, t, hkv, d))
    o = dict(options)
    lens = o.pop("lens", None)
    keys = KeyMask.none() if lens is None else KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device))
    got = svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)), Attn(keys=keys, **o))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, causal=o.get("causal", False), window=o.get("window"),
                                                      key_lens=None if lens is None else np.asarray(lens)))
    # bf16 probabilities and results of values below 1: 2^-8 each way, as in the other oracle tests.
    assert max_abs(to_np(got), want) < 2e-2
