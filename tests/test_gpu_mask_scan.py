"""A key mask row is scanned up front, its 64-key blocks dealt to the waves: rows of every count of blocks at which the deal or
the words' reading turns (a wave's two early blocks, eight in flight, 64 words a read, 256 blocks scanned at most), with
prefixes, holes, single keys and nothing visible, as bytes and as words, against the float64 softmax."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, bits, max_abs, tallies, tally, tally_values, to_np

pytestmark = pytest.mark.gpu


def rows_of(tk):
    """Visibility rows that take each way through the scan."""
    at = np.arange(tk)
    cuts = sorted({1, tk // 3 + 1, 64, 65, 128, 512, 513, max(tk - 1, 1), tk} & set(range(1, tk + 1)))
    rows = [at < n for n in cuts]
    rows += [at >= tk // 2, at == tk - 1, at != 0, (at % 3 != 0), at < 0, (at < tk // 4) | (at >= tk - 2)]
    rows.append(at // 64 % 2 == 0)  # whole blocks shown and hidden in turn
    return np.stack(rows)


KINDS = [
    (7, False, torch.bool), (64, False, torch.int32), (129, True, torch.bool), (256, False, torch.bool), (257, False, torch.int32),
    (512, True, torch.bool), (577, False, torch.bool), (640, False, torch.int32), (2111, False, torch.bool), (2500, False, torch.int32),
    (4096, False, torch.bool), (4097, False, torch.bool), (9001, False, torch.int32), (16384, False, torch.bool),
    (16385, False, torch.bool)]


@pytest.mark.parametrize("tk,causal,kind", KINDS)
def test_every_way_through_the_scan(device, tk, causal, kind):
    mask = rows_of(tk)
    if tk > 4000:
        mask = mask[::3]
    b, h, d = len(mask), 2, 64
    t = tk if causal else 5
    g = Lcg(tk)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, 1, d)), g.bf16((b, tk, 1, d))
    dev = [bf16_tensor(x, device) for x in (q, k, v)]
    shown = torch.from_numpy(mask).to(device)
    keys = KeyMask.bool(shown if kind == torch.bool else shown.to(kind) * 3)
    got = svod_amd.attention(*dev, Attn(causal=causal, keys=keys, splits=1))
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v, causal=causal, key_mask=mask))
    assert np.isfinite(to_np(got)).all() and max_abs(to_np(got), want) < 2e-2
    # A prefix is a length, bit for bit.
    lens = mask.sum(1)
    prefix = (mask == (np.arange(tk)[None, :] < lens[:, None])).all(1)
    as_lens = svod_amd.attention(*dev, Attn(causal=causal, keys=KeyMask.lens(torch.tensor(lens, dtype=torch.int32, device=device)),
                                            splits=1))
    if tk <= 16384:
        assert np.array_equal(bits(got)[prefix], bits(as_lens)[prefix])


@pytest.mark.parametrize("tk,causal,kind", KINDS)
def test_every_key_of_every_block_counts(device, tk, causal, kind):
    """Which keys each row saw, one a column or, of long rows, a block a column: a lost word, a swapped one or a single key shows
    at every length."""
    mask = rows_of(tk)
    if tk > 4000:
        mask = mask[::3] if tk < 16000 else mask[-7:]
    b, d, per = len(mask), 64, 1 if tk <= 640 else 64
    t = tk if causal else 5
    v = tally_values(tk, d, per, device)
    heads = v.shape[2]
    v = v.expand(b, -1, -1, -1).contiguous()
    k = torch.ones(b, tk, 1, d, dtype=torch.bfloat16, device=device).expand(-1, -1, heads, -1).contiguous()
    q = torch.zeros(b, t, heads, d, dtype=torch.bfloat16, device=device)
    shown = torch.from_numpy(mask).to(device)
    keys = KeyMask.bool(shown if kind == torch.bool else shown.to(kind) * 3)
    visible = np.repeat(mask[:, None], t, 1)
    if causal:
        visible = visible & (np.arange(tk)[None, :] <= np.arange(t)[:, None])
    want = tally(visible, d, per)
    got = to_np(svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys, splits=1)))
    assert tallies(got, want)
    # What the bar is for: a row that shows keys, its last visible one hidden, and its last whole block.
    row = int(np.argmax([m.sum() * (m != (np.arange(tk) < m.sum())).any() for m in mask]))
    for lost in (np.flatnonzero(mask[row])[-1:], np.arange(tk) // 64 == np.flatnonzero(mask[row])[-1] // 64):
        other = visible[row, -1].copy()
        other[lost] = False
        assert not tallies(tally(other, d, per), want[row, -1])
