"""Segmented calls whose output segments hold several transition segments
(`per` of the plan, tests/test_seg_plan.py), with and without a remainder, from
a given state and from zero, against the float64 oracle on sampled heads.
Every head has its own inputs, and both ends of the batch are sampled, so a
state taken from another segment or head shows.  rtol = atol = 1e-2 (bf16) and
1e-3 (fp32), as the shorter segmented calls."""
from __future__ import annotations

import pytest
import torch

from oracle import deltanet as odn
from tests.helpers import assert_close
from tests.test_gpu_chain_rec import _inputs
from theorem_amd import chain, configs
from theorem_amd.kernels import _capi, chunk_fwd_h

pytestmark = pytest.mark.gpu

# (kind, B, H, NT, K, V): plans 8 x 2 x 8, 9 x 2 x 7 (17 transition segments of
# 119 chunks), 11 x 2 x 6 (21 of 122, 125: the last output segment has one), 6 x 2 x 10.
FWD = [(1, 16, 128, 128, 128), (1, 13, 119, 128, 128), (2, 5, 122, 64, 128)]
H_BF16 = [(1, 16, 128, 128, 128), (1, 14, 119, 128, 128), (1, 11, 125, 64, 128)]
H_F32 = [(3, 11, 120, 128, 128)]


def np_(t):
    return None if t is None else t.detach().double().cpu().numpy()


@pytest.mark.parametrize("state", [False, True])
@pytest.mark.parametrize("B,H,NT,K,V", FWD)
def test_forward(dev, B, H, NT, K, V, state):
    T = 64 * NT
    q, k, v, beta, a, h0 = _inputs(B, T, H, K, V, NT, dev, 0.1 if state else 0.0)
    scale = K ** -0.5
    o, ht = chain.chunk_gated_delta_rule_fwd(q, k, v, beta, None, scale, h0, True, a=a)
    g = chain.chunk_local_cumsum(a)
    A = chain.build_A(k, beta, g)
    for b, hh in ((0, 0), (B - 1, H - 1)):
        def pick(t):
            return None if t is None else np_(t[b:b + 1, :, hh:hh + 1])
        e0 = None if h0 is None else np_(h0[b:b + 1, hh:hh + 1])
        ew, eu = odn.recompute_w_u_ref(*(pick(t) for t in (k, v, beta, A, g)))
        eh, evn, eht = odn.chunk_fwd_h_delta(pick(k), ew, eu, pick(g), h0=e0)
        eo = odn.chunk_fwd_o_diff(pick(q), pick(k), evn, pick(g), eh, scale)
        assert_close(o[b:b + 1, :, hh:hh + 1], eo, 1e-2, 1e-2, f"o of ({b}, {hh})")
        assert_close(ht[b:b + 1, hh:hh + 1], eht, 1e-2, 1e-2, f"final state of ({b}, {hh})")


@pytest.mark.parametrize("state", [False, True])
@pytest.mark.parametrize("dt,B,H,NT,K,V", [(torch.bfloat16, *s) for s in H_BF16] + [(torch.float32, *s) for s in H_F32])
def test_delta_form(dev, dt, B, H, NT, K, V, state):
    T = 64 * NT
    assert _capi.load_library().thm_chunk_fwd_h_workspace(B, T, H, K, V, _capi.THM_DTYPE[dt], 1) > 0
    d = configs.make_h_inputs(B, T, H, K, V, seed=NT, device=dev, dtype=dt, gate="mild", h0_std=0.1)
    h0 = d.pop("h0")
    if not state:
        h0 = None
    got = chunk_fwd_h.custom_kernel(dict(d, initial_state=h0, output_final_state=True))
    tol = 1e-2 if dt == torch.bfloat16 else 1e-3
    for b, hh in ((0, 0), (B - 1, H - 1)):
        e0 = None if h0 is None else np_(h0[b:b + 1, hh:hh + 1])
        exp = odn.chunk_fwd_h_delta(*(np_(d[n][b:b + 1, :, hh:hh + 1]) for n in ("k", "w", "u", "g")), h0=e0)
        h, vn, ht = (got[0][b:b + 1, :, hh:hh + 1], got[1][b:b + 1, :, hh:hh + 1], got[2][b:b + 1, hh:hh + 1])
        for name, x, e in (("h", h, exp[0]), ("v_new", vn, exp[1]), ("final state", ht, exp[2])):
            assert_close(x, e, tol, tol, f"{name} of ({b}, {hh})")


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("delta", [True, False])
def test_capture(dev, dt, delta):
    # Neither the segments nor the reference form's scan keep anything between
    # calls: a captured call replays to the eager result.
    B, T, H, K, V = (1, 64 * 100, 3, 128, 128) if delta else (2, 64 * 16, 3, 64, 64)
    d = configs.make_h_inputs(B, T, H, K, V, seed=5, device=dev, dtype=dt, gate="mild", h0_std=0.1)
    h0, w, u = d.pop("h0"), d.pop("w"), d.pop("u")
    assert (_capi.load_library().thm_chunk_fwd_h_workspace(B, T, H, K, V, _capi.THM_DTYPE[dt], int(delta)) > 0) == delta
    d.update(dict(w=w, u=u) if delta else dict(v=u), initial_state=h0, output_final_state=True)
    run = lambda: chunk_fwd_h.custom_kernel(d)  # noqa: E731
    ref = run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        for x in got:
            x.zero_()
        graph.replay()
        eager = run()
        torch.cuda.synchronize()
        assert all(torch.equal(x, y) for x, y in zip(ref, got))
        assert all(torch.equal(x, y) for x, y in zip(ref, eager))
