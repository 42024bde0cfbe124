"""GPU parity of chunk_fwd_h's segmented delta form (thm_chunk_fwd_h_ws): every
output against the float64 oracle and against thm_chunk_fwd_h (one piece) on
the same inputs.  rtol = atol = 1e-2 (bf16) and 1e-3 (fp32, whose products
carry ~2^-16); the error may not exceed the one-piece form's by half (P S + Q
is formed in exact fp32 products)."""
from __future__ import annotations

import pytest
import torch

from oracle import deltanet as odn
from tests.helpers import assert_close
from theorem_amd import configs
from theorem_amd.kernels import _capi, chunk_fwd_h

pytestmark = pytest.mark.gpu


def np_(t):
    return None if t is None else t.detach().double().cpu().numpy()


def _one_piece(d, h0, dt):
    k, u = d["k"], d["u"]
    B, T, H, K = k.shape
    V = u.shape[-1]
    h = torch.empty(B, T // 64, H, K, V, device=k.device)
    vn, ht = torch.empty_like(u), torch.empty(B, H, K, V, device=k.device)
    st = _capi.load_library().thm_chunk_fwd_h(
        k.data_ptr(), d["w"].data_ptr(), u.data_ptr(), _capi.ptr(d["g"]), _capi.ptr(h0), h.data_ptr(), vn.data_ptr(),
        ht.data_ptr(), B, T, H, K, V, 64, _capi.THM_DTYPE[dt], 1, _capi.stream_of(k))
    assert st == 0
    return h, vn, ht


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,NT,H,K,V,gated", [(1, 73, 2, 128, 128, True), (1, 71, 3, 128, 64, True),
                                              (2, 67, 2, 64, 128, True), (1, 100, 1, 64, 64, False),
                                              (1, 90, 9, 128, 128, True)])
def test_segments_vs_oracle_and_one_piece(dev, dt, B, NT, H, K, V, gated):
    T = 64 * NT
    assert _capi.load_library().thm_chunk_fwd_h_workspace(B, T, H, K, V, _capi.THM_DTYPE[dt], 1) > 0
    d = configs.make_h_inputs(B, T, H, K, V, seed=NT, device=dev, dtype=dt, gate="mild", h0_std=0.1)
    if not gated:  # without decay: keep the state bounded through w
        d["g"] = None
        d["w"] = (d["k"].float() * 0.05).to(dt)
    h0 = d.pop("h0")
    got = chunk_fwd_h.custom_kernel(dict(d, initial_state=h0, output_final_state=True))
    one = _one_piece(d, h0, dt)
    torch.cuda.synchronize()
    g = d["g"] if gated else torch.zeros(B, T, H)
    exp = odn.chunk_fwd_h_delta(np_(d["k"]), np_(d["w"]), np_(d["u"]), np_(g), h0=np_(h0))
    tol = 1e-2 if dt == torch.bfloat16 else 1e-3
    for name, x, y, e in zip(("h", "v_new", "final state"), got, one, exp):
        what = f"{name} {dt} B={B} NT={NT} H={H} K={K} V={V}"
        assert_close(x, e, tol, tol, what)
        e = torch.from_numpy(e)
        err, err1 = (float((t.double().cpu() - e).norm() / e.norm()) for t in (x, y))
        print(f"{what}: relative error {err:.3e}, in one piece {err1:.3e}")
        assert err <= 1.5 * err1, f"{what}: {err:.3e} against {err1:.3e} in one piece"


def test_optional_outputs_and_refusals(dev):
    d = configs.make_h_inputs(1, 64 * 73, 2, 128, 128, seed=1, device=dev, gate="mild")
    d.pop("h0")
    h, vn, ht = chunk_fwd_h.custom_kernel(dict(d, output_final_state=True))
    h2, vn2, ht2 = chunk_fwd_h.custom_kernel(dict(d, save_new_value=False))
    assert vn2 is None and ht2 is None and torch.equal(h, h2)
    lib = _capi.load_library()
    n = lib.thm_chunk_fwd_h_workspace(1, 64 * 73, 2, 128, 128, 1, 1)
    ws = torch.empty(n, dtype=torch.uint8, device=dev)

    def call(p, nb):
        return lib.thm_chunk_fwd_h_ws(d["k"].data_ptr(), d["w"].data_ptr(), d["u"].data_ptr(), d["g"].data_ptr(), None,
                                      h.data_ptr(), vn.data_ptr(), ht.data_ptr(), p, nb, 1, 64 * 73, 2, 128, 128, 64, 1,
                                      1, _capi.stream_of(h))
    assert call(ws.data_ptr(), n - 1) == -6 and call(None, n) == -1 and call(ws.data_ptr() + 8, n) == -5
    assert call(ws.data_ptr(), n) == 0
    torch.cuda.synchronize()
    # The reference form and filled grids need none.
    assert lib.thm_chunk_fwd_h_workspace(1, 64 * 73, 2, 128, 128, 1, 0) == 0
    assert lib.thm_chunk_fwd_h_workspace(8, 8192, 16, 128, 128, 1, 1) == 0
