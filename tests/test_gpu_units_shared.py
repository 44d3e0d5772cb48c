"""Either side of the lines at which a launch shares its last round of (batch, KV head) pairs out over the XCDs: under eight pairs,
under 48 of more than 128 workgroups, and more, or none left, where it deals them whole.  Every row of every head is written
once, whichever is dealt."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, max_abs, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("key_tiles")]

# (b, t, tk, h, hkv, d, options): pairs x workgroups a pair
CASES = [
    (1, 1100, 70, 15, 15, 32, {}), (1, 1024, 70, 15, 15, 32, {}),            # 15 x 9 shared, 15 x 8 whole
    (3, 1900, 70, 3, 3, 64, {"lens": [70, 1, 40]}),                          # 9 x 15 shared
    (1, 1400, 1400, 12, 12, 64, {"window": (64, 64)}), (1, 1200, 1200, 12, 12, 64, {"window": (64, 64)}),  # 12 x 11, 12 x 10
    (47, 300, 65, 1, 1, 64, {}), (49, 300, 65, 1, 1, 64, {}), (48, 300, 65, 1, 1, 64, {}),
    (3, 400, 100, 15, 5, 128, {}),                                           # 15 x 12, a group's heads in one pair
    (1, 1100, 90, 15, 15, 256, {}), (17, 1000, 66, 1, 1, 48, {}),
    (7, 200, 300, 1, 1, 64, {"lens": [300, 0, 7, 64, 65, 299, 128]}),        # seven pairs
    (9, 40, 100, 3, 1, 64, {}), (130, 40, 100, 3, 1, 64, {}),                # a workgroup a pair
]


@pytest.mark.parametrize("b,t,tk,h,hkv,d,options", CASES, ids=[f"{c[0]}x{c[1]}x{c[2]} {c[3]}/{c[4]}x{c[5]} {' '.join(c[6])}" for c in CASES])
def test_pairs_are_computed_once_each(device, b, t, tk, h, hkv, d, options):
    g = Lcg(19)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, hkv, d)), g.bf16((b, tk, hkv, d))
    o = dict(options)
    lens = o.pop("lens", None)
    keys = KeyMask.none() if lens is None else KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device))
    out = torch.full((b, t, h, d), float("nan"), dtype=torch.bfloat16, device=device)
    got = to_np(svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)), Attn(keys=keys, splits=1, **o), out=out))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, window=o.get("window"), key_lens=None if lens is None else np.asarray(lens)))
    # bf16 probabilities and results of values below 1: 2^-8 each way, as in the other oracle tests.
    assert np.isfinite(got).all() and max_abs(got, want) < 2e-2
