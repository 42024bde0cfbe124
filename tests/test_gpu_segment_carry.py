"""The state crosses segments (chunk records, thm_chunk_fwd_h_ws) as it crosses
chunks in one piece: in fp32.  Where no chunk changes it (beta = 0, or w = u =
0, no gate) every P is the identity and every Q zero, so the state stays h0 to
the last bit."""
from __future__ import annotations

import pytest
import torch

from theorem_amd import chain
from theorem_amd.kernels import _capi, chunk_fwd_h

pytestmark = pytest.mark.gpu

SHAPES = [(1, 41, 3, 128, 64), (2, 37, 2, 64, 128), (1, 100, 1, 64, 64), (1, 128, 16, 128, 128)]


def _randn(gen, dev, *shape):
    return torch.randn(*shape, generator=gen).to(dev)


@pytest.mark.parametrize("B,NT,H,K,V", SHAPES)
def test_forward(dev, B, NT, H, K, V):
    T = 64 * NT
    lib = _capi.load_library()
    assert lib.thm_chunk_gated_delta_rule_workspace(B, T, H, K, V) > B * H * NT * 11 * 1024
    gen = torch.Generator().manual_seed(NT)
    q, k = (_randn(gen, dev, B, T, H, K).bfloat16() for _ in range(2))
    v, h0 = _randn(gen, dev, B, T, H, V).bfloat16(), _randn(gen, dev, B, H, K, V)
    _, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, torch.zeros(B, T, H, device=dev), None, 1.0, h0, True)
    assert torch.equal(ht, h0)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,NT,H,K,V", SHAPES)
def test_delta_form(dev, dt, B, NT, H, K, V):
    T = 64 * NT
    assert _capi.load_library().thm_chunk_fwd_h_workspace(B, T, H, K, V, _capi.THM_DTYPE[dt], 1) > 0
    gen = torch.Generator().manual_seed(NT)
    k, h0 = _randn(gen, dev, B, T, H, K).to(dt), _randn(gen, dev, B, H, K, V)
    w, u = torch.zeros_like(k), torch.zeros(B, T, H, V, dtype=dt, device=dev)
    h, vn, ht = chunk_fwd_h.custom_kernel(dict(k=k, w=w, u=u, g=None, initial_state=h0, output_final_state=True))
    assert torch.equal(h, h0[:, None].expand_as(h)) and torch.equal(ht, h0) and not vn.any()
