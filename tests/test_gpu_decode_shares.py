"""Decoder steps whose rows share the launch's key splits out by their lengths (four splits a row and more over a large cache,
no count named): every distribution of lengths against the float64 softmax, with a cache's row map, appended rows and 64-bit
integers, and a captured step whose lengths, and with them every row's splits, change between its replays."""
import pytest
import torch

import svod_amd
from svod_amd import Attn, Cache, KeyMask
from util import bits

pytestmark = pytest.mark.gpu

# (batch, heads, KV heads, head size, cached keys), and the splits that such a step takes where it names no count.
SHAPES = [(16, 16, 8, 128, 1700), (16, 20, 20, 64, 1300), (4, 16, 8, 128, 6200),
          (17, 8, 4, 128, 2900), (33, 4, 2, 128, 3000), (64, 4, 2, 64, 3200)]  # a lane a row: past 16 and 32 lanes, all 64
UNASKED = [4, 6, 16, 15, 15, 4]


def lengths(kind, b, tk):
    at = torch.arange(b)
    return {"even": torch.full((b,), tk), "wide": 1 + at * (tk - 1) // (b - 1), "one": torch.where(at == b - 2, tk, 3),
            "none": torch.zeros(b), "some": torch.where(at % 3 == 0, tk - at, 0), "short": at % 40,
            "past": torch.full((b,), 2 * tk)}[kind].long()


def tensors(device, b, h, hkv, d, tk, app=0, dtype=torch.bfloat16):
    g = torch.Generator(device=device).manual_seed(b + tk)
    rand = lambda *s: torch.randn(s, generator=g, device=device).to(dtype)
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
    # One rounding to 16 bits (half of 2^-8 of a bf16 value, of 2^-11 of an f16 one) and f32 sums of at most 6300 terms, far
    # below that.
    ulp, rest = (2.0 ** -8, 2.0 ** -12) if got.dtype == torch.bfloat16 else (2.0 ** -11, 2.0 ** -14)
    return ((got.double() - want).abs() <= ulp * want.abs() + rest).all()


@pytest.mark.parametrize("b,h,hkv,d,tk", SHAPES)
@pytest.mark.parametrize("kind", ["even", "wide", "one", "none", "some", "short", "past"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_rows_of_any_lengths(device, b, h, hkv, d, tk, kind, dtype):
    q, k, v = tensors(device, b, h, hkv, d, tk, dtype=dtype)
    lens = lengths(kind, b, tk)
    got = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device, torch.int32))))
    assert close(got, exact(q, k, v, lens))
    wide = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device))))
    assert (bits(wide) == bits(got)).all()


@pytest.mark.parametrize("b,h,hkv,d,tk,unasked", [(*s, n) for s, n in zip(SHAPES, UNASKED)] +
                         [(65, 4, 2, 64, 3200, 7), (16, 16, 8, 128, 1300, 4), (3, 16, 8, 128, 8500, 10)])
def test_which_steps_share(device, b, h, hkv, d, tk, unasked):
    """A step that shares its splits out sums rows of different lengths in other pieces than the same count for every row does,
    which shows in some of its thousands of results; one that does not (more rows than lanes, a cache under 96 MiB, too few
    rows) has that count's bits.  So the cases above run the kernel that they are about."""
    q, k, v = tensors(device, b, h, hkv, d, tk, dtype=torch.float16)
    for integers in (torch.int32, torch.int64):
        keys = KeyMask.lens(lengths("wide", b, tk).to(device, integers))
        got = svod_amd.attention(q, k, v, Attn(keys=keys))
        named = svod_amd.attention(q, k, v, Attn(keys=keys, splits=unasked))
        assert (bits(got) != bits(named)).any() == ((b, h, hkv, d, tk) in SHAPES)


@pytest.mark.parametrize("b,h,hkv,d,tk", SHAPES)
def test_a_row_map_and_appended_rows(device, b, h, hkv, d, tk):
    q, k, v, ka, va = tensors(device, b, h, hkv, d, tk, 3)
    lens, rows, seen = lengths("wide", b, tk).flip(0), torch.randperm(b), torch.arange(b) % 4
    cache = Cache(0, hkv, rows.to(device, torch.int32), appended=(ka, va), app_lens=seen.to(device, torch.int32))
    got = svod_amd.attention(q, k, v, Attn(keys=KeyMask.lens(lens.to(device, torch.int32)), cache=cache))
    assert close(got, exact(q, k, v, lens, rows, (ka, va), seen))


@pytest.mark.parametrize("b,h,hkv,d,tk", [SHAPES[0], SHAPES[5]])
def test_a_captured_step_whose_lengths_change(device, b, h, hkv, d, tk):
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
