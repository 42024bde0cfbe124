"""GPU parity of the whole chunked forward in one call
(thm_chunk_gated_delta_rule_fwd, theorem_amd.chain.chunk_gated_delta_rule_fwd's
bf16 default): chunk records, segment transitions and the output kernel.

Against the float64 oracle (oracle/deltanet.py), rtol = atol = 1e-2 as the
other bf16 paths, and against chunk_fwd_fused_a on the same inputs (A from the
A-builder, the recurrence in one piece), whose error it may not exceed by more
than half: both round S to bf16 inside every chunk, the segments also the columns
of P; P S + Q itself is formed in fp32.
"""
from __future__ import annotations

import pytest
import torch

from oracle import deltanet as odn
from tests.helpers import assert_close
from theorem_amd import chain, configs
from theorem_amd.kernels import _capi

pytestmark = pytest.mark.gpu
REC_BYTES = 11 * 1024


def np_(t):
    return None if t is None else t.detach().double().cpu().numpy()


def _inputs(B, T, H, K, V, seed, dev, h0_std=0.1):
    gen = torch.Generator().manual_seed(seed)
    q = configs.l2norm(torch.randn(B, T, H, K, generator=gen)).to(torch.bfloat16)
    k = configs.l2norm(torch.randn(B, T, H, K, generator=gen)).to(torch.bfloat16)
    v = torch.randn(B, T, H, V, generator=gen).to(torch.bfloat16)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=gen))
    a = -0.02 * torch.rand(B, T, H, generator=gen) - 0.001  # e^{g_last} ~ 0.5: the carry spans many chunks
    h0 = torch.randn(B, H, K, V, generator=gen) * h0_std if h0_std > 0 else None
    to = lambda t: None if t is None else t.to(dev).contiguous()  # noqa: E731
    return to(q), to(k), to(v), to(beta), to(a), to(h0)


def _segmented(B, T, H, K, V):
    n = _capi.load_library().thm_chunk_gated_delta_rule_workspace(B, T, H, K, V)
    assert n >= B * H * (T // 64) * REC_BYTES
    return n > B * H * (T // 64) * REC_BYTES


# One and two chunks; a ragged last segment (37, 41 and 100 chunks); a batch;
# more workgroups than segments pay for.
@pytest.mark.parametrize("B,NT,H,K,V,segmented", [
    (1, 1, 1, 64, 64, False), (2, 2, 3, 128, 128, False), (2, 5, 3, 64, 128, False),
    (1, 37, 2, 128, 128, True), (1, 41, 3, 128, 64, True), (2, 37, 2, 64, 128, True),
    (1, 100, 1, 64, 64, True), (1, 3, 80, 128, 128, False)])
def test_forward_vs_oracle_and_one_piece(dev, B, NT, H, K, V, segmented):
    T = 64 * NT
    assert _segmented(B, T, H, K, V) == segmented
    q, k, v, beta, a, h0 = _inputs(B, T, H, K, V, 7 + NT, dev, 0.1 if NT != 2 else 0.0)
    scale = K ** -0.5
    o, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, scale, h0, True, a=a)
    g = chain.chunk_local_cumsum(a)
    A = chain.build_A(k, beta, g)
    o1, _, ht1 = chain.chunk_fwd_fused_a(q, k, v, beta, A, g, scale, h0, True)
    torch.cuda.synchronize()
    ew, eu = odn.recompute_w_u_ref(np_(k), np_(v), np_(beta), np_(A), np_(g))
    eh, evn, eht = odn.chunk_fwd_h_delta(np_(k), ew, eu, np_(g), h0=np_(h0))
    eo = odn.chunk_fwd_o_diff(np_(q), np_(k), evn, np_(g), eh, scale)
    what = f"B={B} NT={NT} H={H} K={K} V={V}"
    assert_close(o, eo, 1e-2, 1e-2, f"o {what}")
    assert_close(ht, eht, 1e-2, 1e-2, f"final state {what}")
    for name, x, y, e in (("o", o, o1, eo), ("final state", ht, ht1, eht)):
        e = torch.from_numpy(e)
        err, err1 = ((t.double().cpu() - e).norm() / e.norm() for t in (x, y))
        print(f"{what} {name}: relative error {err:.3e}, in one piece {err1:.3e}")
        assert err <= 1.5 * err1, f"{name} {what}: {err:.3e} against {err1:.3e} in one piece"


@pytest.mark.parametrize("NT", [3, 40])
def test_gate_inputs(dev, NT):
    # Every form of the gate gives what the cumsum kernel and the fused forward
    # give: the in-record sums differ from the kernel's by fp32 rounding of |g|
    # <= 60, 60 2^-24 64 < 3e-4 relative in e^{g_i - g_j}, below bf16 rounding.
    B, T, H, K, V = 1, 64 * NT, 2, 128, 64
    q, k, v, beta, a, h0 = _inputs(B, T, H, K, V, 5, dev)
    raw = torch.randn(B, T, H, generator=torch.Generator().manual_seed(6)).to(dev)
    for x, logsig in ((a, False), (a.bfloat16(), False), (raw, True), (raw.bfloat16(), True)):
        g = chain.chunk_local_cumsum(x, logsigmoid=logsig)
        o1, _, ht1 = chain.chunk_fwd_fused_a(q, k, v, beta, chain.build_A(k, beta, g), g, 0.1, h0, True)
        for o, ht in (chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 0.1, h0, True, a=x, a_logsigmoid=logsig),
                      chain.chunk_gated_delta_rule_fwd(q, k, v, beta, g, 0.1, h0, True)):
            assert_close(o, np_(o1), 1e-2, 1e-2, f"o {x.dtype} logsig={logsig}")
            assert_close(ht, np_(ht1), 1e-2, 1e-2, f"final state {x.dtype} logsig={logsig}")
    A = chain.build_A(k, beta, None)
    o1, _, _ = chain.chunk_fwd_fused_a(q, k, v, beta, A, None, 0.1, h0)
    o, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 0.1, h0)
    assert ht is None
    assert_close(o, np_(o1), 1e-2, 1e-2, "o without a gate")


def test_strided_inputs_and_empty(dev):
    B, T, H, K, V = 2, 128, 3, 64, 64
    q, k, v, beta, a, h0 = _inputs(B, T, H, K, V, 9, dev)
    ref = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 0.1, h0, True, a=a)
    strided = [torch.stack([t, t], dim=-1)[..., 0] for t in (q, k, v, beta, a, h0)]
    assert not strided[0].is_contiguous()
    got = chain.chunk_gated_delta_rule_fwd(*strided[:4], None, 0.1, strided[5], True, a=strided[4])
    assert all(torch.equal(x, y) for x, y in zip(ref, got))
    e = chain.chunk_gated_delta_rule_fwd(q[:, :0], k[:, :0], v[:, :0], beta[:, :0], None, 0.1, h0, True, a=a[:, :0])
    assert e[0].shape == (B, 0, H, V) and torch.equal(e[1], h0)


def test_capture(dev):
    # No state between calls: a captured forward replays to the eager result.
    B, T, H, K, V = 1, 64 * 40, 2, 128, 128
    q, k, v, beta, a, h0 = _inputs(B, T, H, K, V, 11, dev)
    run = lambda: chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, 0.1, h0, True, a=a)  # noqa: E731
    ref = run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        got[0].zero_()
        got[1].zero_()
        graph.replay()
        eager = run()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(ref, got))
        assert all(torch.equal(x, y) for x, y in zip(ref, eager))
