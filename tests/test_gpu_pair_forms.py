"""Which calls take a tile's keys in two halves, told by `chosen()`, and every form of operand that they accept: views of a fused
projection, an order of the rows, 64-bit lengths, a bound batch, memory past the lengths that is no number, a captured call,
threads.  Sides without keys are heads of their own here: a group's few queries go side by side in a tile that keeps its keys whole."""
import threading

import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn, Cache, KeyMask
from util import Lcg, bf16_tensor, bits, max_abs, to_np

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("key_tiles")]
SIDES = "sides: 2"


def operands(device, b, t, tk, h, hkv, d, seed=37, f16=False):
    g = Lcg(seed)
    host = tuple(g.bf16(s) for s in ((b, t, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))
    return host, tuple(bf16_tensor(x, device).to(torch.float16 if f16 else torch.bfloat16) for x in host)


def near(host, got, heads=None, **options):
    """Within bf16 probabilities and results of values below 1, 2^-8 each way, of the exact softmax; the named heads alone where
    heads of one KV head are computed alike."""
    q, k, v = host
    heads = list(range(q.shape[2])) if heads is None else heads
    kv = [i * k.shape[2] // q.shape[2] for i in heads]
    p = oracle.AttnProblem(*(np.ascontiguousarray(x) for x in (q[:, :, heads], k[:, :, kv], v[:, :, kv])), **options)
    got = to_np(got)[:, :, heads]
    return bool(np.isfinite(got).all()) and max_abs(got, oracle.attention_direct(p)) < 2e-2


# (b, t, tk, h, hkv, d, causal, options, two sides)
LINES = [
    (1, 130, 513, 2, 2, 64, False, {}, True), (1, 130, 512, 2, 2, 64, False, {}, False),        # over eight key blocks
    (2, 2048, 640, 8, 8, 64, False, {}, True), (2, 2049, 640, 8, 8, 64, False, {}, False),      # 256 workgroups, 272
    (1, 1536, 1536, 32, 8, 128, True, {}, True),                                                # 384 causal, of 12 tiles a head
    (1, 1408, 1408, 32, 8, 128, True, {}, False), (3, 1536, 1536, 16, 8, 128, True, {}, False),  # of 11; 576
    (1, 1536, 1536, 32, 8, 64, True, {}, False), (1, 2100, 600, 16, 16, 128, False, {}, False),  # d 64; 272 not causal
    (1, 130, 600, 2, 2, 64, False, {"splits": 1}, False), (1, 130, 600, 2, 2, 32, False, {}, False),
    (1, 130, 600, 2, 2, 256, False, {}, False), (1, 130, 600, 2, 2, 64, False, {"window": (64, 64)}, False),
    (1, 20, 600, 8, 2, 64, False, {}, False),                                                   # a group in one tile
]


@pytest.mark.parametrize("b,t,tk,h,hkv,d,causal,options,sides", LINES,
                         ids=[f"{c[0]}x{c[1]}x{c[2]} {c[3]}/{c[4]}x{c[5]}{' causal' if c[6] else ''} {' '.join(c[7])}" for c in LINES])
def test_the_lines_of_the_rule(device, b, t, tk, h, hkv, d, causal, options, sides):
    host, (q, k, v) = operands(device, b, t, tk, h, hkv, d)
    got = svod_amd.attention(q, k, v, Attn(causal=causal, **options))
    assert (SIDES in svod_amd.chosen()) == sides, svod_amd.chosen()
    assert near(host, got, [0, h - 1], causal=causal, window=options.get("window"))


def test_a_cache_and_a_bias_keep_the_keys_whole(device):
    _, (q, k, v) = operands(device, 1, 130, 600, 2, 2, 64)
    svod_amd.attention(q, k, v, Attn(cache=Cache(0, 2)))
    assert SIDES not in svod_amd.chosen()
    bias = torch.zeros(1, 2, 130, 600, dtype=torch.bfloat16, device=device)
    svod_amd.attention(q, k, v, Attn(bias=bias))
    assert SIDES not in svod_amd.chosen()


@pytest.mark.parametrize("f16", [False, True], ids=["bf16", "f16"])
@pytest.mark.parametrize("d,causal,t", [(64, False, 33), (64, True, 600), (128, False, 150), (128, True, 577)])
@pytest.mark.parametrize("how", ["lens", "lens64", "bool", "int32"])
def test_rows_that_leave_a_side_nothing(device, d, causal, t, how, f16):
    tk, lens = 600, [600, 0, 1, 64, 65, 320, 321]
    b = len(lens)
    host, (q, k, v) = operands(device, b, t, tk, 1, 1, d, f16=f16)
    n = torch.tensor(lens, dtype=torch.int64 if how == "lens64" else torch.int32, device=device)
    shown = torch.arange(tk, device=device)[None, :] < n[:, None]
    keys = KeyMask.lens(n) if how.startswith("lens") else KeyMask.bool(shown if how == "bool" else shown.to(torch.int32))
    for side in (k, v):  # what no row sees is no number
        for row, count in enumerate(lens):
            if how.startswith("lens"):
                side[row, count:] = float("nan")
    got = svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys))
    assert SIDES in svod_amd.chosen(), svod_amd.chosen()
    assert near(host, got, causal=causal, key_lens=np.asarray(lens))
    assert not bits(got[1]).any()


@pytest.mark.parametrize("h,hkv,d,causal", [(4, 4, 64, False), (8, 2, 64, True), (4, 2, 128, True), (3, 3, 128, False)])
def test_a_fused_projection_read_in_place(device, h, hkv, d, causal):
    b, t = 2, 650
    x = bf16_tensor(Lcg(43).bf16((b, t, (h + 2 * hkv) * d)), device)
    lens = torch.tensor([650, 300], dtype=torch.int32, device=device)
    got = svod_amd.attention_packed(x, h, hkv, Attn(causal=causal, keys=KeyMask.lens(lens)))
    assert SIDES in svod_amd.chosen(), svod_amd.chosen()
    q, k, v = (y.contiguous() for y in x.view(b, t, h + 2 * hkv, d).split([h, hkv, hkv], dim=2))
    assert np.array_equal(bits(got), bits(svod_amd.attention(q, k, v, Attn(causal=causal, keys=KeyMask.lens(lens)))))
    assert near(tuple(to_np(y) for y in (q, k, v)), got, [0, h - 1], causal=causal, key_lens=lens.cpu().numpy())


def test_an_order_of_the_rows_and_a_bound_batch(device):
    host, (q, k, v) = operands(device, 5, 140, 600, 2, 2, 64)
    lens = torch.tensor([100, 600, 0, 599, 300], dtype=torch.int32, device=device)
    keys = KeyMask.lens(lens)
    plain = svod_amd.attention(q, k, v, Attn(keys=keys))
    order = torch.tensor([3, 0, 4, 1, 2], dtype=torch.int32, device=device)
    assert np.array_equal(bits(svod_amd.attention(q, k, v, Attn(keys=keys, row_order=order))), bits(plain))
    assert SIDES in svod_amd.chosen()
    out = torch.full_like(q, 7.0)
    svod_amd.attention(q, k, v, Attn(keys=keys, batch_live=3), out=out)
    assert SIDES in svod_amd.chosen()
    assert np.array_equal(bits(out[:3]), bits(plain[:3])) and bool((out[3:] == 7.0).all())
    assert near(host, plain, key_lens=lens.cpu().numpy())


def test_a_captured_call_replays(device):
    _, (q, k, v) = operands(device, 2, 300, 700, 4, 4, 64)
    lens = torch.tensor([700, 333], dtype=torch.int32, device=device)
    out = torch.empty_like(q)
    opts = Attn(keys=KeyMask.lens(lens))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        svod_amd.attention(q, k, v, opts, out=out)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        svod_amd.attention(q, k, v, opts, out=out)
    assert SIDES in svod_amd.chosen()
    for counts in ([700, 333], [10, 700], [0, 64], [700, 333]):
        lens.copy_(torch.tensor(counts, dtype=torch.int32))
        eager = svod_amd.attention(q, k, v, opts)
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(bits(out), bits(eager)), counts


def test_threads_side_by_side(device):
    cases = [(2, 300, 700, 4, 4, 64, False), (1, 600, 600, 8, 2, 128, True), (3, 130, 577, 2, 2, 128, False)]
    held = [operands(device, *c[:6], seed=50 + i)[1] for i, c in enumerate(cases)]
    want = [bits(svod_amd.attention(*held[i], Attn(causal=c[6]))) for i, c in enumerate(cases)]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                got = [svod_amd.attention(*held[i], Attn(causal=cases[i][6])) for _ in range(30)]
                assert SIDES in svod_amd.chosen()
                stream.synchronize()
            for y in got:
                assert np.array_equal(bits(y), want[i]), i
        except Exception as e:  # noqa: BLE001 - reported by the parent
            errors.append((i, repr(e)))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(cases))]
    for x in threads:
        x.start()
    for x in threads:
        x.join()
    assert not errors, errors
