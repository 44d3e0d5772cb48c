"""The decoder step's workgroups take up to four neighbouring KV heads and a row's splits its chunks in turn: every count of
heads together (which the call's size sets), chunks that end on and off a row's length, appended rows of more than a
chunk, both workgroup sizes, against the float64 softmax (the bars of tests/test_gpu_decode.py)."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, Cache, KeyMask
from util import Lcg, bf16_tensor, bits, max_abs, mean_rel, to_np

pytestmark = pytest.mark.gpu

# (batch, KV heads, group, head size, keys, splits, appended rows).  A chunk is 8192 / (head size * heads together) keys in
# workgroups of four waves: four heads of 64 together 16 keys, two of 128 16, one of 64 64.
CASES = [
    (64, 8, 1, 64, 70, 2, 17),    # four heads of 64, 256 workgroups
    (33, 12, 2, 64, 97, 3, 0),    # four of twelve heads, two rows each, a split for each third chunk
    (48, 6, 1, 64, 49, 2, 64),    # two of six heads: 288 workgroups, 576 of one head
    (64, 5, 1, 64, 66, 2, 1),     # an odd count of heads: one a workgroup
    (33, 16, 2, 128, 50, 1, 33),  # two heads of 128, unsplit
    (32, 16, 1, 128, 130, 3, 3),
    (64, 16, 1, 32, 140, 1, 2),   # four heads of 32
    (40, 8, 1, 48, 90, 4, 20),    # four heads of 48: 384 bytes of a row
    (2, 4, 2, 64, 300, 5, 40),    # eight waves a workgroup
    (3, 2, 1, 256, 100, 2, 9),
    (300, 2, 1, 256, 21, 1, 0),   # a head of 256 is 512 bytes by itself
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,hkv,group,d,tk,splits,n", CASES)
def test_heads_together_over_every_chunk_edge(device, b, hkv, group, d, tk, splits, n, dtype):
    layers, cache_rows, h = 2, 5, hkv * group
    g = Lcg(b + d)
    q, k, v = g.bf16((b, 1, h, d)), g.bf16((cache_rows, tk, layers * hkv, d)), g.bf16((cache_rows, tk, layers * hkv, d))
    lens = np.array([[tk, 0, 1, 15, 16, 17, 31, 32, 33, 63, 64, 65, tk - 1][i % 13] for i in range(b)]).clip(0, tk)
    row_map = np.arange(b) * 3 % cache_rows
    dev = lambda x: bf16_tensor(x, device).to(dtype)
    ints = lambda a: torch.tensor(a, dtype=torch.int32, device=device)
    app = seen = None
    if n:
        app, seen = (g.bf16((b, n, hkv, d)), g.bf16((b, n, hkv, d))), np.array([[n, 0, 1, n - 1][i % 4] for i in range(b)])
        lens[(lens == 0) & (seen == 0)] = 1
    cache = Cache(hkv, hkv, ints(row_map), tuple(dev(x) for x in app) if n else None, ints(seen) if n else None)
    call = lambda keys: svod_amd.attention(dev(q), dev(k), dev(v), Attn(keys=keys, splits=splits, cache=cache))
    got = call(KeyMask.lens(ints(lens)))
    assert "streamed" in svod_amd.chosen() or "combine_splits" in svod_amd.chosen()
    p = oracle.AttnProblem(q, k, v, key_lens=lens, cache=oracle.Cache(hkv, hkv, row_map, app, seen))
    want = oracle.attention_direct(p)
    assert np.isfinite(to_np(got)).all()
    assert max_abs(to_np(got), want) < 2e-2 and mean_rel(to_np(got), want) < 2e-3
    if not n:  # a mask that shows the same keys (with appended rows a call takes lengths alone): another loop
        shown = torch.arange(tk, device=device)[None, :] < ints(lens)[:, None]
        masked = to_np(call(KeyMask.bool(shown)))
        assert max_abs(masked, want) < 2e-2 and mean_rel(masked, want) < 2e-3


@pytest.mark.parametrize("splits", [4, 5, 8, 9, 16, 17, 33, 64])
def test_any_count_of_splits_over_heads_together(device, splits):
    b, hkv, d, tk = 64, 8, 64, 64 * 65
    g = Lcg(splits)
    q, k, v = g.bf16((b, 1, hkv, d)), g.bf16((2, tk, hkv, d)), g.bf16((2, tk, hkv, d))
    rows = np.arange(b) % 2
    lens = np.array([[tk, 70, 0, tk - 1][i % 4] for i in range(b)])
    ints = lambda a: torch.tensor(a, dtype=torch.int32, device=device)
    got = svod_amd.attention(bf16_tensor(q, device), bf16_tensor(k, device), bf16_tensor(v, device),
                             Attn(keys=KeyMask.lens(ints(lens)), splits=splits, cache=Cache(0, hkv, ints(rows))))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, key_lens=lens, cache=oracle.Cache(0, hkv, rows)))
    assert max_abs(to_np(got), want) < 2e-2 and mean_rel(to_np(got), want) < 2e-3


@pytest.mark.parametrize("b,h,hkv,d,tk,rule,better", [
    (16, 16, 8, 128, 2100, 4, 4),   # 512 of two heads: one round of 256 workgroups
    (16, 20, 20, 64, 1500, 3, 6),   # 80 workgroups of four heads a split: 480 are two rounds, nearly full
    (1, 16, 8, 128, 8000, 31, 32),  # more than 16 splits of two heads: 32 of one
    (34, 16, 8, 128, 570, 2, 3),
    (1, 16, 16, 64, 1000, 4, 8),    # 16 KiB of keys a head and split
    (14, 20, 20, 256, 1865, 4, 4),  # 280 (batch, KV head)s: four splits fill seven eighths of five rounds
    (25, 16, 16, 128, 1770, 3, 5),
    (3, 1, 1, 64, 7237, 28, 16),    # as many as one trip of the merge takes
    (2, 2, 2, 128, 16000, 62, 32),
    (15, 20, 20, 64, 576, 2, 3),    # heads together, rather than four splits of one head
    (27, 20, 20, 64, 530, 2, 4),    # nor three
    (4, 16, 16, 64, 1481, 6, 8),    # nor twelve
    (22, 12, 12, 48, 1014, 4, 3)])  # nor six
def test_the_count_that_a_step_takes_unasked(device, b, h, hkv, d, tk, rule, better):
    """The rule's with the workspace that it asks for, or the device's own where that is less, which twice as much always takes."""
    g = torch.Generator(device=device).manual_seed(b)
    q, k, v = (torch.randn(s, generator=g, device=device).bfloat16() for s in ((b, 1, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))
    named = lambda n: bits(svod_amd.attention(q, k, v, Attn(splits=n)))
    assert np.array_equal(bits(svod_amd.attention(q, k, v)), named(better))
    lent = torch.empty(rule * b * h * (d + 2) * 4 + 128 * b * hkv, dtype=torch.uint8, device=device)
    assert np.array_equal(bits(svod_amd.attention(q, k, v, workspace=lent)), named(min(rule, better)))
    out = torch.empty_like(q)
    assert np.array_equal(bits(svod_amd.attention_noalloc(q, k, v, Attn(), out)), named(better))


@pytest.mark.parametrize("b,h,hkv,d,tk", [(64, 8, 8, 128, 1024), (32, 16, 16, 128, 1024), (60, 8, 8, 128, 1024), (25, 20, 20, 64, 600)])
def test_a_step_splits_when_a_workspace_is_asked_for(device, b, h, hkv, d, tk):
    """What svodk_attention_workspace answers is what the call does, given that much and in the package's own."""
    g = torch.Generator(device=device).manual_seed(b)
    q, k, v = (torch.randn(s, generator=g, device=device).bfloat16() for s in ((b, 1, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))
    need = svod_amd.ops._calls().attention_workspace(q, k, Attn())
    lent = torch.empty(max(need, 16), dtype=torch.uint8, device=device)
    for workspace in (lent, None):
        got = svod_amd.attention(q, k, v, workspace=workspace)
        assert ("combine_splits" in svod_amd.chosen()) == (need > 0)
        whole = svod_amd.attention(q, k, v, Attn(splits=1))
        assert mean_rel(to_np(got), to_np(whole)) < 2e-3
        if need == 0:
            assert np.array_equal(bits(got), bits(whole))
