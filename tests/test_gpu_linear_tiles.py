"""The projection GEMM's tiles at the sizes where each can go wrong: rows and columns on and off the tile, k in whole
and half lines and shared out unevenly over eight waves, turned heads of both sizes, a bias, both types, a window of a
wider output.  Against the unrounded f64 epilogue at the reference's bar (tk/src/test/unit/ops.rs:312)."""
import numpy as np
import pytest
import torch

import oracle
import svod_amd
from svod_amd import Linear, Rotary
from util import Lcg, assert_rel_close, bf16_tensor, mean_rel

pytestmark = pytest.mark.gpu

# (rows, n, k, head size turned or 0, heads turned, bias, f16) -> the tile the shape takes
CASES = [
    ((1, 8, 512, 0, 0, True, False), (16, 16)),
    ((16, 4096, 544, 128, 24, False, False), (16, 16)),
    ((17, 200, 1024, 64, 3, True, True), (16, 16)),
    ((33, 584, 832, 0, 0, True, False), (16, 16)),
    ((30, 4096, 512, 64, 40, True, False), (32, 16)),
    ((32, 2320, 608, 0, 0, False, True), (32, 16)),
    ((45, 3072, 576, 128, 23, True, False), (32, 32)),
    ((64, 4096, 512, 64, 1, False, True), (32, 32)),
    ((100, 2304, 768, 64, 24, True, False), (64, 32)),
    ((127, 4040, 512, 0, 0, True, False), (64, 32)),
    ((250, 2304, 544, 128, 17, True, False), (64, 64)),
    ((193, 4096, 512, 64, 33, False, True), (64, 64)),
    ((257, 4032, 544, 64, 60, True, False), (128, 64)),
    ((512, 4096, 512, 0, 0, False, True), (128, 64)),
    ((300, 4096, 512, 128, 31, True, False), (128, 128)),
    ((1, 40, 32, 0, 0, True, False), (128, 128)),
    ((129, 392, 96, 64, 5, True, True), (128, 128)),
    ((2400, 4096, 96, 0, 0, True, False), (256, 192)),
    ((2305, 3976, 64, 0, 0, False, True), (256, 192)),
    ((3600, 4096, 64, 128, 24, True, False), (256, 256)),
    ((3585, 4040, 96, 64, 60, False, True), (256, 256)),
]


@pytest.mark.parametrize("case,tile", CASES, ids=["x".join(str(int(v)) for v in c[0]) for c in CASES])
def test_each_tile_matches_the_reference(device, case, tile):
    rows, n, k, d, heads, bias, f16 = case
    g = Lcg(rows * 31 + n)
    dtype, rounded = (torch.float16, oracle.round_f16) if f16 else (torch.bfloat16, oracle.round_bf16)
    up = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dtype).to(device)
    x, w, bv = (rounded(a) for a in (g.bf16((1, rows, k)), g.bf16((n, k), mul=0.3), g.bf16((n,))))
    opts, rope = {"bias": up(bv)} if bias else {}, None
    if d:
        cos, sin = (rounded(a) for a in oracle.rope_table(10_000.0, rows, d))
        opts["rope"] = Rotary(*(up(a.reshape(1, rows, 1, d // 2)) for a in (cos, sin)), heads, d)
        rope = (cos, sin, heads, d)
    wide = torch.full((1, rows, n + 24), 3.0, dtype=dtype, device=device)
    svod_amd.linear(up(x), up(w), Linear(into=(wide, 8), **opts))
    torch.cuda.synchronize()
    assert "bm: %d, bn: %d," % tile in svod_amd.chosen(), svod_amd.chosen()
    assert bool((wide[..., :8] == 3.0).all()) and bool((wide[..., 8 + n:] == 3.0).all())
    got = wide[0, :, 8:8 + n].float().cpu().numpy()
    # Every row where there are few, else the tiles' edges and a spread: the oracle sums in f64 on the host.
    at = np.arange(rows) if rows * n * k < 6e8 else np.unique(np.r_[0:3, 126:130, 254:258, rows - 130:rows - 126, rows - 3:rows, 500:rows:517])
    at = at[at < rows]
    pick = (rope[0][at], rope[1][at], heads, d) if rope else None
    want = oracle.linear_direct(x[:, at], w, bv if bias else None, pick)[0]
    assert_rel_close(str(case), got[at], want, 2e-2)
    assert mean_rel(got[at], rounded(want.astype(np.float32))) < 3e-4
