"""Launches of at most one workgroup a compute unit over nine key blocks and more run eight waves a tile, two sides of four
that take half of the key blocks each and merge in LDS: odd counts of blocks, sides that a length, a causal edge or the end
of the keys leaves nothing, scales of either sign, and both sides of the line."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, max_abs, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("key_tiles")]

# (b, t, tk, h, hkv, d, causal, lens, scale, dtype)
CASES = [
    (1, 130, 512, 2, 2, 64, False, None, None, "bf16"),              # eight key blocks: the last in four waves
    (1, 130, 513, 2, 2, 64, False, None, None, "bf16"),              # nine: five and four
    (1, 1, 700, 3, 1, 128, False, [700], None, "bf16"),              # a query
    (7, 33, 640, 2, 1, 64, False, [640, 0, 1, 64, 320, 321, 65], None, "bf16"),  # sides without keys
    (6, 200, 577, 2, 2, 128, False, [577, 576, 63, 0, 128, 129], None, "f16"),
    (1, 530, 530, 2, 2, 64, True, None, None, "bf16"),               # causal: tiles of two to nine
    (3, 600, 600, 2, 1, 128, True, [600, 5, 300], None, "bf16"),
    (2, 257, 700, 2, 2, 64, True, [700, 100], None, "f16"),          # more keys than queries see
    (1, 700, 577, 2, 2, 128, True, None, None, "bf16"),              # fewer
    (2, 100, 600, 2, 2, 64, False, [600, 70], -0.11, "bf16"),        # the maximum in the exponent's units
    (1, 100, 600, 2, 2, 128, False, None, 0.0, "bf16"),              # every key the same
    (2, 2048, 640, 8, 8, 64, False, [640, 77], None, "bf16"),        # 256 workgroups
    (2, 2049, 640, 8, 8, 64, False, [640, 77], None, "bf16"),        # 272: four waves
    (1, 1536, 1536, 32, 4, 128, True, None, None, "bf16"),           # 384 of 12 tiles a head
]


@pytest.mark.parametrize("b,t,tk,h,hkv,d,causal,lens,scale,dtype", CASES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]} {c[3]}/{c[4]}x{c[5]}{' causal' if c[6] else ''} {c[9]}" for c in CASES])
def test_two_sides_of_a_tile_are_one(device, b, t, tk, h, hkv, d, causal, lens, scale, dtype):
    g = Lcg(23)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, hkv, d)), g.bf16((b, tk, hkv, d))
    keys = KeyMask.none() if lens is None else KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device))
    cast = (lambda x: bf16_tensor(x, device)) if dtype == "bf16" else (lambda x: bf16_tensor(x, device).to(torch.float16))
    got = to_np(svod_amd.attention(*(cast(x) for x in (q, k, v)), Attn(causal=causal, keys=keys, scale=scale)).to(torch.float32))
    # Heads of one KV head are computed alike, so the oracle takes the first and the last alone.
    ends = sorted({0, h - 1})
    kv = [i * hkv // h for i in ends]
    want = oracle.attention_direct(oracle.AttnProblem(
        np.ascontiguousarray(q[:, :, ends]), np.ascontiguousarray(k[:, :, kv]), np.ascontiguousarray(v[:, :, kv]),
        causal=causal, scale=scale, key_lens=None if lens is None else np.asarray(lens)))
    # bf16 probabilities and results of values below 1: 2^-8 each way, as in the other oracle tests.
    assert np.isfinite(got).all() and max_abs(got[:, :, ends], want) < 2e-2
    if lens is not None and 0 in lens:
        assert not got[lens.index(0)].any()
