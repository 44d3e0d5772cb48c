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
    """An eager step's last workgroup merges, a captured step launches the merge: the same bits, call after call and
    with other streams' steps beside it."""
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
