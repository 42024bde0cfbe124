"""Segmented forwards on sequences far from contractive: a segment's map
overflows fp32 while the states stay finite (zero, or off the growing
direction).  The results are the recurrence's, as in one piece."""
from __future__ import annotations

import pytest
import torch

from theorem_amd import chain
from theorem_amd.kernels import _capi, chunk_fwd_h

pytestmark = pytest.mark.gpu

SHAPES = [(1, 41, 3, 128, 64), (2, 37, 2, 64, 128), (1, 128, 16, 128, 128)]


def _h0(B, H, K, V, dev):
    """Zero along dimension 0, the direction that k grows; zero in the first columns."""
    h0 = torch.randn(B, H, K, V, generator=torch.Generator().manual_seed(3)).to(dev)
    h0[:, :, 0] = 0
    h0[..., :20] = 0
    return h0


@pytest.mark.parametrize("B,NT,H,K,V", SHAPES)
def test_forward(dev, B, NT, H, K, V):
    # Every token scales dimension 0 by 1 - beta |k|^2 = -3: 3^64 a chunk, past fp32 in two.
    T = 64 * NT
    lib = _capi.load_library()
    assert lib.thm_chunk_gated_delta_rule_workspace(B, T, H, K, V) > B * H * NT * 11 * 1024
    k = torch.zeros(B, T, H, K, dtype=torch.bfloat16, device=dev)
    k[..., 0] = 2.0
    q = torch.zeros_like(k)
    q[..., 1] = 1.0
    v, beta, h0 = torch.zeros(B, T, H, V, dtype=torch.bfloat16, device=dev), torch.ones(B, T, H, device=dev), _h0(B, H, K, V, dev)
    o, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 1.0, h0, True)
    assert torch.equal(ht, h0)
    assert torch.equal(o, h0[:, None, :, 1].expand(B, T, H, V).bfloat16())
    o, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 1.0, None, True)
    assert not o.any() and not ht.any()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,NT,H,K,V", SHAPES)
def test_delta_form(dev, dt, B, NT, H, K, V):
    # A chunk scales dimension 0 by 1 + 64 * 2^43 ~ 6e14, past fp32 in three.
    # Only the last chunk has u: v_new = u there, its k^T u ends up in row 0.
    # One head's k is zero: its segments' maps stay finite beside the others.
    T = 64 * NT
    assert _capi.load_library().thm_chunk_fwd_h_workspace(B, T, H, K, V, _capi.THM_DTYPE[dt], 1) > 0
    k = torch.zeros(B, T, H, K, dtype=dt, device=dev)
    k[:, :, :-1, 0] = 1.0
    w, u = -(2.0 ** 43) * k, torch.zeros(B, T, H, V, dtype=dt, device=dev)
    u[:, -64:, :, : V // 2] = 0.5
    h0 = _h0(B, H, K, V, dev)
    h, vn, ht = chunk_fwd_h.custom_kernel(dict(k=k, w=w, u=u, g=None, initial_state=h0, output_final_state=True))
    last = h0.clone()
    last[:, :-1, 0, : V // 2] = 32.0
    assert torch.equal(h, h0[:, None].expand_as(h)) and torch.equal(vn, u) and torch.equal(ht, last)
