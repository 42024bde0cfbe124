"""The host fast path of the conv decode step, the channels-last conv and the
chunked forward: bit-identical to the ctypes path, and None (the ctypes path,
with its errors) outside the common case.  The one-sample kernel of the decode
step against the general one over widths and state lengths."""
from __future__ import annotations

import pytest
import torch

from theorem_amd import chain
from theorem_amd.kernels import _capi, causal_conv1d

pytestmark = pytest.mark.gpu


def _both(fn, monkeypatch):
    fast = fn()
    with monkeypatch.context() as m:
        m.setattr(_capi, "fastpath", lambda: None)
        slow = fn()
    torch.cuda.synchronize()
    return fast, slow


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("W", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("extra", [0, 1, 3])
@pytest.mark.parametrize("act", [None, "silu"])
def test_update(dev, dtype, W, extra, act, monkeypatch):
    # state_len W - 1 and W take the one-sample kernel, W + 2 the general one;
    # each gives the full-sequence conv's last output and the shifted state.
    B, D, Ls = 3, 301, W - 1 + extra
    gen = torch.Generator().manual_seed(W)
    mk = lambda *n: torch.randn(*n, generator=gen).to(dtype).to(dev)  # noqa: E731
    x, st, w, b = mk(B, D), mk(B, D, Ls), mk(D, W), mk(D)

    def run():
        s = st.clone()
        return causal_conv1d.causal_conv1d_update(x, s, w, b, act), s
    fast, slow = _both(run, monkeypatch)
    assert all(torch.equal(p, q) for p, q in zip(fast, slow))
    seq = torch.cat([st, x.unsqueeze(-1)], dim=-1).contiguous()
    full = causal_conv1d.custom_kernel((seq, w, b), activation=act)
    assert torch.equal(fast[0], full[..., -1]) and torch.equal(fast[1], seq[..., 1:])


def test_channels_last(dev, monkeypatch):
    x = torch.randn(2, 33, 48, device=dev).transpose(1, 2)
    w, b = torch.randn(48, 4, device=dev), torch.randn(48, device=dev)
    fp = _capi.fastpath()
    assert fp.conv1d_channels_last(x, w, b, 0) is not None and fp.conv1d(x, w, b, 0) is None
    assert fp.conv1d_channels_last(x.contiguous(), w, b, 0) is None
    assert fp.conv1d_channels_last(x[:, :, ::2], w, b, 0) is None
    fast, slow = _both(lambda: causal_conv1d.custom_kernel((x, w, b)), monkeypatch)
    assert torch.equal(fast, slow) and fast.stride() == slow.stride() == x.stride()
    with pytest.raises(AssertionError):
        causal_conv1d.custom_kernel((x[:, :, ::2], w, b))


def test_forward(dev, monkeypatch):
    B, T, H, K, V = 2, 128, 3, 64, 128
    mk = lambda *n: torch.randn(*n, device=dev)  # noqa: E731
    q, k, v = (0.1 * mk(B, T, H, n) for n in (K, K, V))
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    beta, a, h0 = torch.sigmoid(mk(B, T, H)), -0.1 * torch.rand(B, T, H, device=dev), mk(B, H, K, V)
    for want in (False, True):
        fast, slow = _both(lambda: chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 0.1, h0, want, a=a), monkeypatch)
        assert torch.equal(fast[0], slow[0])
        assert torch.equal(fast[1], slow[1]) if want else fast[1] is None and slow[1] is None
    fp = _capi.fastpath()
    assert fp.gated_delta_rule(q, k, v, beta, a, 0, h0, 0.1, True) is not None
    assert fp.gated_delta_rule(q.float(), k, v, beta, a, 0, h0, 0.1, True) is None
    assert fp.gated_delta_rule(q, k, v, beta.bfloat16(), a, 0, h0, 0.1, True) is None
    assert fp.gated_delta_rule(q[:, :100], k[:, :100], v[:, :100], beta[:, :100], None, 0, h0, 0.1, True) is None
    with pytest.raises(AssertionError):
        chain.chunk_gated_delta_rule_fwd(q.float(), k, v, beta, None, 0.1, a=a)
    with pytest.raises(AssertionError):
        chain.chunk_gated_delta_rule_fwd(q, k, v, beta.bfloat16(), None, 0.1, a=a)
