"""Host-side checks of thm_chunk_gated_delta_rule_fwd: a call that the C side
refuses launches nothing (no GPU needed), in the codes of the entry points it
composes."""
from __future__ import annotations

import pytest

from theorem_amd.kernels import _capi


def call(q=16, k=16, v=16, beta=16, gate=16, h0=None, o=16, ht=16, ws=16, nws=1 << 40, B=1, T=128, H=2, K=64, V=64,
         bt=64, dt=1, gdt=0, kind=0):
    return _capi.load_library().thm_chunk_gated_delta_rule_fwd(q, k, v, beta, gate, h0, o, ht, ws, nws, 1.0, B, T, H,
                                                               K, V, bt, dt, gdt, kind, None)


@pytest.mark.parametrize("kw,status", [
    (dict(q=None), -1), (dict(k=None), -1), (dict(v=None), -1), (dict(beta=None), -1), (dict(o=None), -1),
    (dict(ws=None), -1), (dict(T=100), -2), (dict(B=-1), -2), (dict(H=0), -2), (dict(B=1 << 32), -2),
    (dict(dt=0), -3), (dict(gdt=2), -3), (dict(gdt=1, kind=2), -3), (dict(K=96), -4), (dict(V=32), -4),
    (dict(H=1 << 20, T=64), -4), (dict(q=8), -5), (dict(ws=8), -5), (dict(o=4), -5), (dict(beta=2), -5),
    (dict(gate=2), -5), (dict(bt=32), -6), (dict(kind=3), -6), (dict(nws=100), -6),
])
def test_refused(kw, status):
    assert call(**kw) == status


def test_nothing_to_do():
    assert call(B=0) == 0 and call(T=0, ht=None) == 0


def test_workspace():
    ws = _capi.load_library().thm_chunk_gated_delta_rule_workspace
    assert ws(1, 64, 1, 64, 64) == 11 * 1024 and ws(0, 64, 1, 64, 64) == 0 and ws(1, 0, 1, 64, 64) == 0
    assert ws(1, 100, 1, 64, 64) < 0 and ws(1, 64, 1, 96, 64) < 0
