"""Windows and chunks of which a wave's 32 rows see none of the tile's first key blocks: the wave comes past those blocks and
scores its own first one behind them.  Edges one key to either side of a block's, rows no key is left for, splits, and segment
starts that fall within a wave, against the float64 softmax."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, max_abs, tallies, tally, tally_values, to_np

pytestmark = pytest.mark.gpu


def saw(device, visible, d, opts):
    """The call's keys, one a column, are those of `visible` [b, t, tk] for each query."""
    b, t, tk = visible.shape
    v = tally_values(tk, d, 1, device)
    heads = v.shape[2]
    v = v.expand(b, -1, -1, -1).contiguous()
    q = torch.zeros(b, t, heads, d, dtype=v.dtype, device=device)
    got = to_np(svod_amd.attention(q, torch.ones_like(v), v, opts))
    want = tally(visible, d, 1)
    assert (np.isfinite(got)).all() and ((got != 0) == (want != 0)).all() and tallies(got, want)


def in_window(t, tk, window, lens, causal):
    i, j = np.arange(t)[:, None], np.arange(tk)[None, :]
    seen = np.ones((t, tk), bool) if window is None else (j >= i - window[0]) & (j <= i + window[1])
    if causal:
        seen = seen & (j <= i)
    return np.stack([seen & (j < n) for n in lens])


@pytest.mark.parametrize("t,window,lens,splits,causal", [
    (128, (0, 0), None, None, False), (129, (31, 0), None, None, True), (257, (32, 1), None, None, False),
    (300, (63, 63), [300, 17], None, False), (300, (64, 64), [130, 299], None, False), (300, (65, 0), None, None, True),
    (511, (16, 200), [511, 64], 2, False), (512, (127, 3), [500, 0], 3, False), (640, (128, 128), [640, 400], None, True)])
@pytest.mark.parametrize("d", [64, 128])
def test_windows_past_the_first_blocks(device, t, window, lens, splits, causal, d):
    g = Lcg(t + d)
    q, k, v = (g.bf16((2, t, 2, d)) for _ in range(3))
    keys = KeyMask.none() if lens is None else KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device))
    got = svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)),
                             Attn(causal=causal, keys=keys, window=window, splits=splits))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, causal=causal, window=window,
                                                      key_lens=None if lens is None else np.asarray(lens)))
    assert np.isfinite(to_np(got)).all() and max_abs(to_np(got), want) < 2e-2
    saw(device, in_window(t, t, window, lens or [t, t], causal), d,
        Attn(causal=causal, keys=keys, window=window, splits=splits))


@pytest.mark.parametrize("starts", [[0, 40, 70, 200], [0, 96, 130, 131], [0, 200, 10, 64]])
def test_segment_starts_that_turn_within_a_wave(device, starts):
    """One tile of 128 rows, whose first row starts at key 0; the last case's starts fall."""
    t, d = 128, 64
    g = Lcg(len(starts) + starts[1])
    q, k, v = g.bf16((1, t, 2, d)), g.bf16((1, 256, 2, d)), g.bf16((1, 256, 2, d))
    seg = np.repeat(np.asarray(starts), 32)[None].astype(np.int32)
    seg[0, 20:32] = starts[1] if starts[1] < starts[2] else 0
    got = svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)),
                             Attn(seg_start=torch.from_numpy(seg).to(device), window=(500, 500)))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, seg_start=seg, window=(500, 500)))
    assert max_abs(to_np(got), want) < 2e-2
    saw(device, np.arange(256)[None, None, :] >= seg[:, :, None], d, Attn(seg_start=torch.from_numpy(seg).to(device), window=(500, 500)))


@pytest.mark.parametrize("lens,causal", [([1, 32, 33, 64], False), ([65, 96, 97, 128], False), ([31, 95, 129, 200], True)])
@pytest.mark.parametrize("d", [48, 64, 128])
def test_lengths_at_the_edges_of_a_half_block(device, lens, causal, d):
    """A block's half of 32 keys that no row sees is left out, on either side of the diagonal's and of a length's."""
    t = 200 if causal else 70
    g = Lcg(lens[0] + d)
    q, k, v = g.bf16((4, t, 2, d)), g.bf16((4, 200, 2, d)), g.bf16((4, 200, 2, d))
    keys = KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device))
    got = svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)), Attn(causal=causal, keys=keys, splits=1))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, causal=causal, key_lens=np.asarray(lens)))
    assert np.isfinite(to_np(got)).all() and max_abs(to_np(got), want) < 2e-2
    saw(device, in_window(t, 200, None, lens, causal), d, Attn(causal=causal, keys=keys, splits=1))


def test_a_mask_that_shows_one_half_of_every_block(device):
    """Halves shown and hidden in turn, and blocks hidden whole: what is left out is what the mask says."""
    t, d = 40, 64
    g = Lcg(3)
    q, k, v = g.bf16((3, t, 2, d)), g.bf16((3, 384, 2, d)), g.bf16((3, 384, 2, d))
    at = np.arange(384)
    mask = np.stack([at // 32 % 2 == 0, at // 32 % 2 == 1, at // 96 % 2 == 1])
    got = svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)),
                             Attn(keys=KeyMask.bool(torch.from_numpy(mask).to(device)), splits=1))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, key_mask=mask))
    assert max_abs(to_np(got), want) < 2e-2
    saw(device, np.repeat(mask[:, None], t, 1), d, Attn(keys=KeyMask.bool(torch.from_numpy(mask).to(device)), splits=1))
