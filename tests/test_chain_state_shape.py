"""The bf16 forwards refuse an initial_state (or gate) of another shape before any
launch: the kernels would read B H K V floats from its pointer.  The checks come
before the device check, so they are seen on CPU tensors too."""
from __future__ import annotations

import pytest
import torch

from theorem_amd import chain
from theorem_amd.kernels import _capi

B, T, H, K, V = 2, 128, 3, 64, 128
WRONG = [(1, H, K, V), (B, H - 1, K, V), (B, H, V, K), (B, H, K), (B * H, K, V), (B, H, K, V, 1)]


def inputs(device):
    bf = dict(dtype=torch.bfloat16, device=device)
    q, k, w = (torch.zeros(B, T, H, K, **bf) for _ in range(3))
    v = torch.zeros(B, T, H, V, **bf)
    f = torch.zeros(B, T, H, device=device)
    return q, k, w, v, f, torch.zeros(B, T, H, 64, device=device)


def calls(device, h0, g=None):
    q, k, w, v, f, A = inputs(device)
    g = f if g is None else g
    return [lambda: chain.chunk_gated_delta_rule_fwd(q, k, v, f, g, 1.0, initial_state=h0),
            lambda: chain.chunk_gated_delta_rule_fwd(q, k, v, f, None, 1.0, initial_state=h0, a=g),
            lambda: chain.chunk_fwd_fused_a(q, k, v, f, A, g, 1.0, initial_state=h0),
            lambda: chain.chunk_fwd_fused(q, k, w, v, g, 1.0, initial_state=h0)]


def check(device, shape):
    for call in calls(device, torch.zeros(*shape, device=device)):
        with pytest.raises(AssertionError, match="initial_state"):
            call()


@pytest.mark.parametrize("shape", WRONG)
def test_refused(shape):
    check("cpu", shape)


def test_fused_gate_shape():
    """chunk_fwd_fused checks its gate as the other forms do."""
    q, k, w, v, f, _ = inputs("cpu")
    with pytest.raises(AssertionError) as e:
        chain.chunk_fwd_fused(q, k, w, v, torch.zeros(1, T, H), 1.0)
    assert "device" not in str(e.value)


@pytest.mark.gpu
@pytest.mark.parametrize("fast", [True, False], ids=["fast", "python"])
@pytest.mark.parametrize("shape", WRONG)
def test_refused_gpu(shape, fast, monkeypatch):
    if not fast:
        monkeypatch.setattr(_capi, "fastpath", lambda: None)
    check("cuda", shape)
