"""A tile's two sides take its key blocks in turn, so that a key mask which shows a row's first keys is the row's length: the same
blocks for each side, the same bits.  (Halves in a row were cut before the mask was read, and hid a side's whole work.)"""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, bits, max_abs, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("elements", [torch.bool, torch.int32])
@pytest.mark.parametrize("t,h,hkv,d,causal", [(130, 2, 2, 64, False), (700, 2, 2, 64, True), (150, 1, 1, 128, False), (650, 4, 2, 128, True)])
def test_a_padding_mask_is_a_length(device, t, h, hkv, d, causal, elements):
    tk, lens = 700, [700, 699, 640, 577, 385, 384, 130, 128, 127, 65, 64, 1, 0]
    b = len(lens)
    g = Lcg(61)
    q, k, v = (bf16_tensor(g.bf16(s), device) for s in ((b, t, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))
    n = torch.tensor(lens, dtype=torch.int32, device=device)
    for at in (slice(0, 4), slice(4, 8), slice(8, 13)):  # a few rows at a time: a workgroup a compute unit
        by_length = svod_amd.attention(q[at], k[at], v[at], Attn(causal=causal, keys=KeyMask.lens(n[at])))
        assert "sides: 2" in svod_amd.chosen(), svod_amd.chosen()
        shown = (torch.arange(tk, device=device)[None, :] < n[at, None]).to(elements)
        by_mask = svod_amd.attention(q[at], k[at], v[at], Attn(causal=causal, keys=KeyMask.bool(shown)))
        assert "sides: 2" in svod_amd.chosen(), svod_amd.chosen()
        assert np.array_equal(bits(by_mask), bits(by_length))


@pytest.mark.parametrize("tk", [64 * 512, 64 * 512 + 1, 64 * 513, 64 * 513 + 64])
def test_rows_around_what_a_side_scans(device, tk):
    # 256 blocks a side are scanned ahead; with 513 one side scans and the other reads its row a block at a time.
    g = Lcg(67)
    q, k, v = (bf16_tensor(g.bf16((1, n, 1, 64)), device) for n in (40, tk, tk))
    mask = np.arange(tk)[None, :] % 5 != 2
    mask[:, 100:9000] = False
    mask[:, tk - 300:tk - 70] = False
    opts = Attn(keys=KeyMask.bool(torch.from_numpy(mask).to(device)))
    # A lent workspace of a few bytes: the keys are not split.
    got = to_np(svod_amd.attention(q, k, v, opts, workspace=torch.empty(16, dtype=torch.uint8, device=device)))
    assert "sides: 2" in svod_amd.chosen(), svod_amd.chosen()
    want = oracle.attention_direct(oracle.AttnProblem(*(to_np(x) for x in (q, k, v)), key_mask=mask))
    # bf16 probabilities and results of values below 1: 2^-8 each way, as in the other oracle tests.
    assert np.isfinite(got).all() and max_abs(got, want) < 2e-2
