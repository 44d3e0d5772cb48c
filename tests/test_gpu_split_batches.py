"""The merge of key splits takes their states eight at a time: counts at and past a batch's edges."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Attn
from util import Lcg, bf16_tensor, bits, max_abs, mean_rel, to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("splits,d,t", [(7, 64, 1), (8, 32, 1), (9, 128, 2), (16, 64, 5), (17, 48, 1), (33, 256, 1)])
def test_any_count_of_splits_merges_to_the_softmax(device, splits, d, t):
    b, h, tk = 2, 2, 64 * 33 - 5
    g = Lcg(splits)
    q, k, v = g.bf16((b, t, h, d)), g.bf16((b, tk, h, d)), g.bf16((b, tk, h, d))
    got = to_np(svod_amd.attention(*(bf16_tensor(x, device) for x in (q, k, v)), Attn(splits=splits)))
    assert "combine_splits" in svod_amd.chosen()
    want = oracle.attention_direct(oracle.AttnProblem(q, k, v))
    assert max_abs(got, want) < 2e-2
    assert mean_rel(got, oracle.round_bf16(want.astype(np.float32))) < 4e-3


@pytest.mark.parametrize("splits,d,h,hkv,t", [(2, 64, 3, 3, 1), (8, 48, 2, 2, 1), (9, 128, 4, 2, 1), (17, 256, 2, 2, 2), (33, 32, 1, 1, 1)])
def test_a_step_that_merges_its_own_splits_equals_one_that_leaves_them(device, splits, d, h, hkv, t):
    """A step's last workgroup merges where the workspace has room for its words, a launch of its own where it has not
    (the captured one here): the same bits, call after call and with other streams' steps beside it."""
    b, tk = 3, 64 * 33 - 5
    g = Lcg(100 + splits)
    q, k, v = (bf16_tensor(g.bf16(s), device) for s in ((b, t, h, d), (b, tk, hkv, d), (b, tk, hkv, d)))
    opts = Attn(keys=svod_amd.KeyMask.lens(torch.tensor([tk, 70, 0], dtype=torch.int32, device=device)), splits=splits)
    out, ws = torch.empty_like(q), torch.empty(splits * b * t * h * (d + 2) * 4, dtype=torch.uint8, device=device)
    eager = bits(svod_amd.attention(q, k, v, opts))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        svod_amd.attention(q, k, v, opts, out=out, workspace=ws)
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        beside = []
        for s in streams:
            with torch.cuda.stream(s):
                beside += [svod_amd.attention(q, k, v, opts) for _ in range(4)]
        torch.cuda.synchronize()
        assert np.array_equal(bits(out), eager)
        assert all(np.array_equal(bits(x), eager) for x in beside)


def lent(splits, b, t, h, hkv, d, device, merges=True):
    """A workspace of the partial states, and of the words with which a step merges them itself."""
    return torch.empty(splits * b * t * h * (d + 2) * 4 + (128 * b * hkv if merges else 0), dtype=torch.uint8, device=device)


@pytest.mark.parametrize("splits,b,h,hkv,t", [(2, 300, 5, 5, 1), (8, 3, 4, 2, 1), (64, 2, 2, 2, 2), (65, 2, 2, 2, 1)])
def test_a_captured_step_merges_its_own_splits_over_any_content(device, splits, b, h, hkv, t):
    """What the workspace holds does not matter: noise, zeros, ones, the words as the replay before left them.  More than
    64 splits are left to the merge."""
    d, tk = 64, 64 * 65 - 9 if splits >= 64 else 64 * 9
    g = Lcg(200 + splits)
    rows = torch.arange(b, dtype=torch.int32, device=device) % 3
    q = bf16_tensor(g.bf16((b, t, h, d)), device)
    k, v = (bf16_tensor(g.bf16((3, tk, hkv, d)), device) for _ in range(2))
    lens = torch.tensor([[tk, 70, 0, tk - 1][i % 4] for i in range(b)], dtype=torch.int32, device=device)
    opts = Attn(keys=svod_amd.KeyMask.lens(lens), cache=svod_amd.Cache(0, hkv, rows), splits=splits)
    want = bits(svod_amd.attention(q, k, v, opts, workspace=lent(splits, b, t, h, hkv, d, device, merges=False)))
    ws, out = lent(splits, b, t, h, hkv, d, device), torch.empty_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        svod_amd.attention(q, k, v, opts, out=out, workspace=ws)
    noise = torch.randint(0, 256, ws.shape, dtype=torch.uint8, device=device)
    for content in (noise, None, torch.zeros_like(ws), None, torch.full_like(ws, 255), None, None):
        if content is not None:
            ws.copy_(content)
        out.fill_(float("nan"))
        graph.replay()
        assert np.array_equal(bits(out), want)
        out.fill_(float("nan"))
        svod_amd.attention(q, k, v, opts, out=out, workspace=ws)
        assert np.array_equal(bits(out), want)


def test_steps_on_many_streams_that_come_and_go(device):
    """A hundred streams, each destroyed with its step in flight, so that handles come again: the steps share nothing."""
    import ctypes

    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    b, h, d, tk, splits = 4, 8, 64, 2048, 8
    g = Lcg(321)
    q, k, v = (bf16_tensor(g.bf16(s), device) for s in ((b, 1, h, d), (b, tk, h, d), (b, tk, h, d)))
    opts = Attn(splits=splits)
    want = bits(svod_amd.attention(q, k, v, opts, workspace=lent(splits, b, 1, h, h, d, device, merges=False)))
    sets = [(torch.full_like(q, float("nan")), lent(splits, b, 1, h, h, d, device)) for _ in range(100)]
    torch.cuda.synchronize()
    for out, ws in sets:
        handle = ctypes.c_void_p()
        assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
        with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
            svod_amd.attention(q, k, v, opts, out=out, workspace=ws)
        assert hip.hipStreamDestroy(handle) == 0
    torch.cuda.synchronize()
    for out, _ in sets:
        assert np.array_equal(bits(out), want)
