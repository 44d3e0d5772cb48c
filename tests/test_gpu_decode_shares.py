"""Decoder steps whose rows share the launch's key splits out by their lengths (four splits a row and more over a large cache,
no count named): every distribution of lengths against the float64 softmax, with a cache's row map, appended rows and 64-bit
integers, and a captured step whose lengths, and with them every row's splits, change between its replays."""
import pytest
import torch

import svod_amd
from svod_amd import Attn, Cache, KeyMask
from util import bits

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 8, 128, 1700), (16, 20, 20, 64, 1300), (4, 16, 8, 128, 6200)]


def lengths(kind, b, tk):
    at = torch.arange(b)
    return {"even": torch.full((b,), tk), "wide": 1 + at * (tk - 1) // (b - 1), "one": torch.where(at == b - 2, tk, 3),
            "none": torch.zeros(b), "some": torch.where(at % 3 == 0, tk - at, 0), "short": at % 40,
            "past": torch.full((b,), 2 * tk)}[kind].long()


def tensors(device, b, h, hkv, d, tk, app=0):
    g = torch.Generator(device=device).manual_seed(b + tk)
    rand = lambda *s: torch.randn(s, generator=g, device=device).bfloat16()
    return [rand(b, 1, h, d), rand(b, tk, hkv, d), rand(b, tk, hkv, d)] + [rand(b, app, hkv, d) for _ in range(2 if app else 0)]


def exact(q, k, v, lens, rows=None, app=None, app_lens=None):
    """The float64 softmax, a batch row at a time."""
    b, _, h, d = q.shape
    out = torch.zeros(b, 1, h, d, dtype=torch.float64, device=q.device)
    for i in range(b):
        at = i if rows is None else int(rows[i])
        n = min(int(lens[i]), k.shape[1])
        keys, vals = k[at, :n], v[at, :n]
        if app is not None:
            keys, vals = torch.cat([keys, app[0][i, :int(app_lens[i])]]), torch.cat([vals, app[1][i, :int(app_lens[i])]])
        if len(keys) == 0:
            continue
        group = h // k.shape[2]
        keys, vals = (x.double().repeat_interleave(group, 1) for x in (keys, vals))
        p = torch.softmax((keys * q[i].double()).sum(-1) * d ** -0.5, 0)
        out[i, 0] = (p[:, :, None] * vals).sum(0)
    return out


def close(got, want):
    # One rounding to bf16 (half of 2^-8 of the value) and f32 sums of at most 6300 terms, far below that.
    return ((got.double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -12).all()


@pytest.mark.parametrize("b,h,hkv,d,tk", SHAPES)
@pytest.mark.parametrize("kind", ["even", "wide", "one", "none", "some", "short", "past"])
def test_rows_of_any_lengths(device, b, h, hkv, d, tk, kind):
    q, k, v = tensors(device, b, h, hkv, d, tk)
    lens = lengths(kind, b, tk)
    got = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device, torch.int32))))
    assert close(got, exact(q, k, v, lens))
    wide = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device))))
    assert (bits(wide) == bits(got)).all()


@pytest.mark.parametrize("b,h,hkv,d,tk", SHAPES)
def test_a_row_map_and_appended_rows(device, b, h, hkv, d, tk):
    q, k, v, ka, va = tensors(device, b, h, hkv, d, tk, 3)
    lens, rows, seen = lengths("wide", b, tk).flip(0), torch.randperm(b), torch.arange(b) % 4
    cache = Cache(0, hkv, rows.to(device, torch.int32), appended=(ka, va), app_lens=seen.to(device, torch.int32))
    got = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device, torch.int32)), cache=cache))
    assert close(got, exact(q, k, v, lens, rows, (ka, va), seen))


def test_a_captured_step_whose_lengths_change(device):
    b, h, hkv, d, tk = SHAPES[0]
    q, k, v = tensors(device, b, h, hkv, d, tk)
    lens, out = torch.empty(b, dtype=torch.int32, device=device), torch.empty_like(q)
    room = torch.empty(64 << 20, dtype=torch.uint8, device=device)
    opts = Attn(keys=KeyMask.lens(lens))
    call = lambda to: svod_amd.attention(q, k, v, opts, out=to, workspace=room)
    lens.copy_(lengths("even", b, tk))
    call(out)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for kind in ["even", "wide", "one", "even", "some", "none", "wide", "wide"]:
        lens.copy_(lengths(kind, b, tk))
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        replayed = out.clone()
        assert close(replayed, exact(q, k, v, lengths(kind, b, tk))), kind
        eager = torch.empty_like(q)
        call(eager)
        assert (bits(eager) == bits(replayed)).all(), kind
