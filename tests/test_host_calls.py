"""The native side of the Python calls (svod_amd/csrc/host.cpp) on operands it has to refuse itself, before the
library sees them."""
import ctypes
import sys
import weakref

import pytest
import torch

import svod_amd
from svod_amd import Attn, Linear, OpError, Qkv

X = torch.zeros((2, 4, 512), dtype=torch.bfloat16)
W = torch.zeros(512, dtype=torch.bfloat16)
Q = torch.zeros((2, 4, 8, 64), dtype=torch.bfloat16)


@pytest.mark.parametrize("call,kind", [
    (lambda: svod_amd.rms_norm(X.double(), W), "Dtype"),
    (lambda: svod_amd.rms_norm(X[None, None], W), "Shape"),
    (lambda: svod_amd.add_layer_norm(X, X.transpose(0, 1).contiguous().transpose(0, 1), W), "Argument"),
    (lambda: svod_amd.attention(Q, Q, Q[:, ::2]), "Argument"),
    (lambda: svod_amd.attention(Q, Q, Q, Attn(bias=Q.double())), "Dtype"),
    (lambda: svod_amd.attention_packed(X.double(), 2, 2), "Dtype"),
    (lambda: svod_amd.heads(X.double(), Qkv(4, 2, 64)), "Dtype"),
    (lambda: svod_amd.linear(X, torch.zeros((512, 64), dtype=torch.bfloat16).T, Linear()), "Argument"),
    (lambda: svod_amd.order_rows(torch.zeros(4, dtype=torch.uint8)), "Dtype"),
])
def test_operands_without_a_descriptor_are_refused(call, kind):
    with pytest.raises(OpError) as e:
        call()
    assert e.value.kind == kind


@pytest.mark.parametrize("call", [lambda: svod_amd.rms_norm(X, None), lambda: svod_amd.attention(Q, Q, 3)])
def test_what_is_no_tensor_is_a_type_error(call):
    with pytest.raises(TypeError):
        call()


class Computed:
    """Options whose tensors are made when they are asked for, and held by nobody else."""

    def __init__(self, made, **fields):
        self.__dict__.update(_made=made, _fields=fields)

    def __getattr__(self, name):
        x = self._fields[name]
        if not callable(x):
            return x
        x = x()
        self._made += [weakref.ref(t) for t in (x if isinstance(x, tuple) else (x,))]
        return x


def test_a_computed_option_lives_to_the_end_of_the_call():
    """The library is handed addresses: whatever they are of is alive when it is called."""
    native, made, dead = svod_amd.ops._calls(), [], []
    lib = svod_amd.load_library()
    names = ["attention", "attention_noalloc", "attention_packed", "attention_workspace", "heads", "linear", "layer_norm",
             "add_layer_norm", "rms_norm", "add_rms_norm", "order_rows"]
    real = {"svodk_" + n: ctypes.cast(getattr(lib, "svodk_" + n), ctypes.c_void_p).value for n in names}

    def look(*_):
        dead.append(sum(r() is None for r in made))
        return 0

    stand_ins = [ctypes.CFUNCTYPE(ctypes.c_int, *[ctypes.c_void_p] * n)(look) for n in (6, 6, 5)]
    attn, heads, linear = (ctypes.cast(f, ctypes.c_void_p).value for f in stand_ins)
    types = tuple(svod_amd.ops._DTYPES)
    i32 = lambda *shape: (lambda: torch.zeros(shape, dtype=torch.int32))
    b16 = lambda *shape: (lambda: torch.zeros(shape, dtype=torch.bfloat16))
    pair = lambda *shape: (lambda: (b16(*shape)(), b16(*shape)()))
    cache = Computed(made, head_start=0, kv_heads=8, row_map=i32(2), appended=pair(2, 1, 8, 64), app_lens=i32(2))
    a = Computed(made, causal=False, keys=Computed(made, kind=1, tensor=i32(2)), window=None, chunk=None, seg_start=i32(2, 4),
                 cache=cache, bias=b16(2, 8, 4, 5), splits=1, scale=None, batch_live=None, row_order=i32(2))
    qkv = Computed(made, heads=4, kv_heads=2, head_dim=64, q_norm=b16(64), k_norm=b16(64), eps=1e-6, rope=pair(1, 4, 1, 32),
                   batch_live=None)
    rope = Computed(made, cos=b16(1, 4, 1, 32), sin=b16(1, 4, 1, 32), heads=4, head_dim=64)
    lin = Computed(made, bias=b16(512), act=0, gated=False, residual=b16(2, 4, 512), scale=None, rope=rope, batch_live=None, into=None)
    native.bind({**real, "svodk_attention": attn, "svodk_heads": heads, "svodk_linear": linear}, OpError, svod_amd.ops._finish, types)
    try:
        svod_amd.attention(Q, Q, Q, a)
        svod_amd.heads(X, qkv)
        svod_amd.linear(X, torch.zeros((512, 512), dtype=torch.bfloat16), lin)
    finally:
        native.bind(real, OpError, svod_amd.ops._finish, types)
    assert len(made) == 8 + 4 + 4
    # A later call finds the earlier ones' options gone.
    assert dead == [0, 8, 12]


def test_a_missing_native_side_says_how_to_build_it(monkeypatch):
    monkeypatch.setattr(svod_amd.ops, "_native", None)
    monkeypatch.setitem(sys.modules, "svod_amd._host", None)  # what an import that cannot succeed meets
    monkeypatch.delattr(svod_amd, "_host", raising=False)
    with pytest.raises(ImportError, match="python -m svod_amd.build"):
        svod_amd.rms_norm(X, W)


def test_the_build_is_of_everything_that_the_package_loads(monkeypatch):
    from svod_amd import build

    outputs = []
    monkeypatch.setattr(build, "_run", lambda cmd, verbose: outputs.append(cmd[cmd.index("-o") + 1]))
    build.build()
    assert {build.LIB, build.HOST} <= set(outputs)
