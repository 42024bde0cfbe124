"""GPU parity of thm_wy_build_A_gates (A and the cumulative gates in one launch,
fp32) with thm_chunk_local_cumsum and thm_wy_build_A.  The two sum 64 gates in
different orders: each is within 63 * 2^-24 of the sum of magnitudes, so they
differ by at most twice that, and A, given the same g, is the same kernel's."""
from __future__ import annotations

import pytest
import torch

from theorem_amd import chain, configs
from theorem_amd.kernels import _capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,K", [(1, 64, 1, 64), (2, 192, 3, 128), (1, 128, 17, 64)])
@pytest.mark.parametrize("adt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("logsig", [False, True])
def test_A_and_gates(dev, B, T, H, K, adt, logsig):
    gen = torch.Generator().manual_seed(T + H)
    k = configs.l2norm(torch.randn(B, T, H, K, generator=gen)).to(dev)
    v = torch.randn(B, T, H, 64, generator=gen).to(dev)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=gen)).to(dev)
    a = (torch.randn(B, T, H, generator=gen) if logsig else -0.1 * torch.rand(B, T, H, generator=gen)).to(adt).to(dev)
    A, g = chain._build_A_gates(k, beta, a, logsig)
    g0 = chain.chunk_local_cumsum(a, logsigmoid=logsig)
    # Every gate is <= 0, so -g0 is the sum of magnitudes.
    assert bool(((g - g0).abs() <= 126 * 2.0 ** -24 * -g0).all())
    assert torch.equal(A, chain.build_A(k, beta, g))
    o, ht = chain.chunk_gated_delta_rule_fwd(k, k, v, beta, None, 0.1, None, True, a=a, a_logsigmoid=logsig)
    o1, ht1 = chain.chunk_gated_delta_rule_fwd(k, k, v, beta, g, 0.1, None, True)
    assert torch.equal(o, o1) and torch.equal(ht, ht1)


@pytest.mark.parametrize("logsig", [False, True])
def test_intermediates_only_add_outputs(dev, logsig):
    # Asking for the intermediates changes no bit of o and the final state, and
    # the g and A returned are those they were formed from.
    B, T, H, K = 2, 192, 3, 128
    gen = torch.Generator().manual_seed(1)
    k = configs.l2norm(torch.randn(B, T, H, K, generator=gen)).to(dev)
    v = torch.randn(B, T, H, 64, generator=gen).to(dev)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=gen)).to(dev)
    a = (torch.randn(B, T, H, generator=gen) if logsig else -0.1 * torch.rand(B, T, H, generator=gen)).to(dev)
    o, ht = chain.chunk_gated_delta_rule_fwd(k, k, v, beta, None, 0.1, None, True, a=a, a_logsigmoid=logsig)
    o1, ht1, mid = chain.chunk_gated_delta_rule_fwd(k, k, v, beta, None, 0.1, None, True, a=a, a_logsigmoid=logsig,
                                                    return_intermediates=True)
    assert torch.equal(o, o1) and torch.equal(ht, ht1)
    A, g = chain._build_A_gates(k, beta, a, logsig)
    assert torch.equal(mid["A"], A) and torch.equal(mid["g"], g)


def test_refused():
    f = _capi.load_library().thm_wy_build_A_gates
    ok = dict(k=16, beta=16, a=16, A=16, g=16, B=1, T=64, H=1, K=64, bt=64, kd=0, ad=0, kind=0, sign=1)
    for kw, st in ((dict(k=None), -1), (dict(a=None), -1), (dict(g=None), -1), (dict(T=65), -2), (dict(kd=1), -3),
                   (dict(ad=2), -3), (dict(K=96), -4), (dict(k=8), -5), (dict(a=2), -5), (dict(bt=32), -6),
                   (dict(kind=2), -6), (dict(sign=0), -6)):
        x = {**ok, **kw}
        assert f(*x.values(), None) == st, kw
    assert f(*{**ok, "B": 0}.values(), None) == 0
