"""The native side of the Python calls (svod_amd/csrc/host.cpp) on operands it has to refuse itself, before the
library sees them."""
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
