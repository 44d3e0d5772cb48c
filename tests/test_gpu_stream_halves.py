"""The streaming knob changes no bit of any call: those that take a tile's keys in two halves run that form whatever the knob
says, and the others' two forms agree (tests/test_gpu_stream.py)."""
import threading

import numpy as np
import pytest
import torch

import svod_amd
from svod_amd import Attn, KeyMask
from util import Lcg, bf16_tensor, bits

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def automatic_again():
    yield
    svod_amd.tune_streaming(0)


# (b, t, tk, h, hkv, causal, mask): over nine key blocks and more in a workgroup a compute unit or fewer
CASES = [
    (1, 130, 700, 2, 2, False, None), (2, 300, 600, 2, 2, False, "lens"), (2, 700, 700, 4, 2, True, None),
    (3, 200, 577, 3, 1, False, "bool"), (2, 2048, 640, 8, 8, False, "lens"),
    (2, 2049, 640, 8, 8, False, "lens"),  # one workgroup too many
]


def operands(device, b, t, tk, h, hkv, mask):
    g = Lcg(11)
    q, k, v = (bf16_tensor(g.bf16(s), device) for s in ((b, t, h, 64), (b, tk, hkv, 64), (b, tk, hkv, 64)))
    lens = torch.tensor([tk - 50 * i for i in range(b)], dtype=torch.int32, device=device)
    keys = {None: KeyMask.none(), "lens": KeyMask.lens(lens),
            "bool": KeyMask.bool(torch.arange(tk, device=device)[None, :] < lens[:, None])}[mask]
    return q, k, v, keys


@pytest.mark.parametrize("b,t,tk,h,hkv,causal,mask", CASES)
def test_every_setting_gives_the_same_bits(device, b, t, tk, h, hkv, causal, mask):
    q, k, v, keys = operands(device, b, t, tk, h, hkv, mask)
    plain = bits(svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys)))
    for slots in (-1, 2, 96):
        svod_amd.tune_streaming(slots)
        assert np.array_equal(bits(svod_amd.attention(q, k, v, Attn(causal=causal, keys=keys))), plain), slots


def test_a_knob_turned_between_calls_changes_no_bit(device):
    q, k, v, keys = operands(device, 2, 300, 600, 2, 2, "lens")
    plain = bits(svod_amd.attention(q, k, v, Attn(keys=keys)))
    done = threading.Event()

    def turn():
        while not done.is_set():
            for slots in (0, 3, -1, 5):
                svod_amd.tune_streaming(slots)

    turner = threading.Thread(target=turn)
    turner.start()
    try:
        for i in range(100):
            assert np.array_equal(bits(svod_amd.attention(q, k, v, Attn(keys=keys))), plain), i
    finally:
        done.set()
        turner.join()
