"""GPU parity of chunk_fwd_h's reference form where its chunks run side by side
(csrc/chunk_fwd_h_scan.hip) against the float64 oracle: batches of 16 chunks
that are short, whole and followed by a remainder, both tile sizes, one and
two rounds of workgroups, head counts with the plain and the per-XCD mapping,
with and without gates and initial state.

Bounds on the relative error in the 2-norm: bf16 rounds v e^{g_last - g} to
2^-9 of itself (products and sums in fp32); fp32 products are exact and each
element sums 64 products a chunk in fp32, whose errors of 2^-24 grow no faster
than the square root of their count here (random signs): 2^-24 * 8 a chunk
and, as the carry decays or keeps h's own size, 2^-24 a scan step."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import deltanet as odn
from theorem_amd import configs
from theorem_amd.kernels import chunk_fwd_h

pytestmark = pytest.mark.gpu


def np_(t):
    return None if t is None else t.detach().double().cpu().numpy()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,NT,H,K,V,plain", [
    (1, 5, 3, 64, 64, False), (2, 16, 3, 64, 64, False), (1, 17, 1, 128, 128, True), (1, 37, 8, 64, 64, False),
    (1, 33, 1, 64, 128, False),                                     # 16 x 16 tiles
    (1, 5, 9, 128, 128, False), (1, 16, 8, 128, 64, True), (2, 31, 5, 64, 128, False),
    (1, 33, 16, 128, 128, False),                                   # 32 x 32
    (1, 32, 20, 128, 128, False), (1, 31, 20, 128, 128, False),     # two rounds, and walked just below
])
def test_scan_vs_oracle(dev, dt, B, NT, H, K, V, plain):
    d = configs.make_h_inputs(B, 64 * NT, H, K, V, seed=NT, device=dev, dtype=dt, gate="mild", h0_std=0.1)
    g, h0 = (None, None) if plain else (d["g"], d["h0"])
    h, ht = chunk_fwd_h.custom_kernel(dict(k=d["k"], v=d["u"], g=g, initial_state=h0, output_final_state=True))
    alone = chunk_fwd_h.custom_kernel(dict(k=d["k"], v=d["u"], g=g, initial_state=h0))
    torch.cuda.synchronize()
    assert torch.equal(alone, h)
    k, v = np_(d["k"]), np_(d["u"])
    gk = np.zeros((B, 64 * NT, H)) if g is None else np_(g)
    pre, _, eht = odn.chunk_fwd_h_delta(k, np.zeros_like(k), v, gk, h0=np_(h0))
    eh = np.concatenate([pre[:, 1:], eht[:, None]], axis=1)
    bound = 2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -24 * (8 + NT)
    if dt == torch.float32 and NT == 31 and H == 20:
        bound = 2.0 ** -16  # the walking kernel's products of bf16 hi + lo
    for name, x, e in (("h", h, eh), ("final state", ht, eht)):
        err = np.linalg.norm(np_(x) - e) / np.linalg.norm(e)
        assert err <= bound, f"{name}: relative error {err:.3e}, bound {bound:.3e}"


# Heads rounded up to whole rounds of the XCDs: one workgroup per CU (45 heads of
# 4 tiles, 15 of 16), two (45 of 8, 17 of 16).
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,NT,H,K,V", [(5, 17, 9, 64, 64), (1, 6, 15, 128, 128), (5, 32, 9, 128, 64), (1, 33, 17, 128, 128)])
def test_heads_not_a_multiple_of_the_xcds(dev, dt, B, NT, H, K, V):
    test_scan_vs_oracle(dev, dt, B, NT, H, K, V, False)
