"""A tile's two sides under a key mask: each scans its own half of the row's blocks.  Masks that are a length, that have holes,
that leave either side or both nothing, odd counts of blocks, a causal edge, and rows too long for a side to scan."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, max_abs, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("key_tiles")]


def _mask(kind, tk):
    m = np.zeros(tk, dtype=bool)
    if kind == "all":
        m[:] = True
    elif kind == "padded":
        m[:tk - tk // 5 - 7] = True
    elif kind == "short":
        m[:70] = True
    elif kind == "late":
        m[tk - 40:] = True
    elif kind == "holes":
        m[np.arange(tk) % 7 != 3] = True
        m[200:400] = False
    elif kind == "one":
        m[tk // 2 + 1] = True
    return m  # "nothing": all hidden


# (b of kinds, t, tk, h, hkv, d, causal, scale, dtype)
CASES = [
    (["all", "padded", "short", "late", "holes", "one", "nothing"], 33, 640, 2, 1, 64, False, None, "bf16"),
    (["all", "padded", "short", "late", "holes", "one", "nothing"], 150, 577, 1, 1, 128, False, None, "f16"),
    (["padded"], 130, 513, 2, 2, 64, False, None, "bf16"),
    (["holes"], 130, 512, 2, 2, 64, False, None, "bf16"),  # eight key blocks: four waves
    (["all", "holes", "late"], 600, 600, 2, 2, 128, True, None, "bf16"),
    (["padded", "nothing"], 530, 530, 2, 2, 64, True, None, "f16"),
    (["padded", "holes"], 100, 600, 2, 2, 64, False, -0.11, "bf16"),
    (["holes", "padded"], 2048, 640, 8, 8, 64, False, None, "bf16"),  # 256 workgroups
]


@pytest.mark.parametrize("elements", ["bool", "int32"])
@pytest.mark.parametrize("kinds,t,tk,h,hkv,d,causal,scale,dtype", CASES,
                         ids=[f"{len(c[0])}x{c[1]}x{c[2]} {c[3]}/{c[4]}x{c[5]}{' causal' if c[6] else ''} {c[8]}" for c in CASES])
def test_each_side_reads_its_own_half_of_the_mask(device, kinds, t, tk, h, hkv, d, causal, scale, dtype, elements):
    g, b = Lcg(29), len(kinds)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, hkv, d)), g.bf16((b, tk, hkv, d))
    mask = np.stack([_mask(kind, tk) for kind in kinds])
    keys = KeyMask.bool(torch.from_numpy(mask if elements == "bool" else mask.astype(np.int32)).to(device))
    cast = (lambda x: bf16_tensor(x, device)) if dtype == "bf16" else (lambda x: bf16_tensor(x, device).to(torch.float16))
    got = to_np(svod_amd.attention(*(cast(x) for x in (q, k, v)), Attn(causal=causal, keys=keys, scale=scale)).to(torch.float32))
    # Heads of one KV head are computed alike, so the oracle takes the first and the last alone.
    ends = sorted({0, h - 1})
    kv = [i * hkv // h for i in ends]
    want = oracle.attention_direct(oracle.AttnProblem(
        np.ascontiguousarray(q[:, :, ends]), np.ascontiguousarray(k[:, :, kv]), np.ascontiguousarray(v[:, :, kv]),
        causal=causal, scale=scale, key_mask=mask))
    # bf16 probabilities and results of values below 1: 2^-8 each way, as in the other oracle tests.
    assert np.isfinite(got).all() and max_abs(got[:, :, ends], want) < 2e-2
    for row, kind in enumerate(kinds):
        if kind == "nothing":
            assert not got[row].any()


def test_a_row_too_long_for_a_side_to_scan(device):
    tk = 2 * 256 * 64 + 130  # 257 and 258 blocks a side
    g = Lcg(31)
    q, k, v = (bf16_tensor(g.bf16((1, n, 16, 64)), device) for n in (2048, tk, tk))
    mask = torch.from_numpy(_mask("holes", tk)[None]).to(device)
    mask[:, 40:9000] = False
    got, whole = (to_np(svod_amd.attention(q, k, v, Attn(keys=KeyMask.bool(mask), splits=s))) for s in (None, 1))
    # Both lie within the oracle's 2e-2 of the exact result by the tests above; of each other, within their two roundings.
    assert np.isfinite(got).all() and max_abs(got, whole) < 2e-2
