"""Gated DeltaNet chunk forward composed from the three HIP kernels.

    A      = (I + strict_lower(beta_i (k_i . k_j) e^{g_i - g_j}))^{-1}   per 64-token chunk
    (w, u) = recompute_w_u(k, v, beta, A, g)                            HIP
    (h, v_new, S) = chunk_fwd_h delta form (h[c] before chunk c)        HIP
    o      = chunk_fwd_o(q, k, v_new, g, h, scale)                      HIP
    (for bf16 the last three in one kernel from A, chunk_fwd_fused_a, which
    never forms w and u; or the first two in one kernel, wy_fwd, and the last
    two in another, chunk_fwd_fused)

The reference never composes its ops (each is tested alone); this is the
forward of chunked Gated DeltaNet that the three ops are the stages of, and
it reproduces the token-by-token gated delta rule
    S_t = e^{a_t} S_{t-1};  S_t += beta_t k_t (v_t - S_t^T k_t)^T;  o_t = scale S_t^T q_t
with g the chunk-local cumsum of a.

``build_A`` (the WY matrix) is the HIP kernel thm_wy_build_A; ``wy_fwd`` is
thm_wy_fwd.
"""
from __future__ import annotations

import torch

from .kernels import _capi, chunk_fwd_h, chunk_fwd_o, recompute_w_u

BT = 64


def chunk_local_cumsum(a: torch.Tensor, logsigmoid: bool = False) -> torch.Tensor:
    """g [B, T, H] fp32: per 64-token chunk, the inclusive cumsum of a (or of
    log(sigmoid(a)) with ``logsigmoid``), on the GPU (thm_chunk_local_cumsum)."""
    B, T, H = a.shape
    assert T % BT == 0, f"T={T} must be a multiple of {BT}"
    _capi.require_device(a)
    code = _capi.dtype_code(a, "a")
    a = _capi.prep(a, "a")
    g = torch.empty(B, T, H, dtype=torch.float32, device=a.device)
    status = _capi.load_library().thm_chunk_local_cumsum(
        _capi.ptr(a), _capi.ptr(g), B, T, H, BT, code, 1 if logsigmoid else 0, _capi.stream_of(a))
    _capi.check(status, "thm_chunk_local_cumsum")
    return g


def build_A(k: torch.Tensor, beta: torch.Tensor, g: torch.Tensor | None) -> torch.Tensor:
    """A [B, T, H, 64] fp32 = per-chunk (I + strict_lower(beta_i k_i.k_j e^{g_i - g_j}))^{-1} (HIP)."""
    return recompute_w_u.build_A(k, beta, g, sign=+1)


def _check_state(initial_state, B: int, H: int, K: int, V: int) -> None:
    """The kernels read B H K V floats from initial_state, whatever its shape."""
    assert initial_state is None or initial_state.shape == (B, H, K, V), (
        f"initial_state {tuple(initial_state.shape)} must be {(B, H, K, V)}")


def wy_fwd(k: torch.Tensor, v: torch.Tensor, beta: torch.Tensor, g: torch.Tensor | None,
           sign: int = +1) -> tuple[torch.Tensor, torch.Tensor]:
    """(w, u) = recompute_w_u(k, v, beta, A, g) with A = build_A(k, beta, g, sign)
    formed inside the same HIP kernel and never written (thm_wy_fwd; bf16 k, v)."""
    B, T, H, K = k.shape
    V = v.shape[-1]
    assert T % BT == 0, f"T={T} must be a multiple of {BT}"
    assert v.shape[:3] == (B, T, H) and beta.shape == (B, T, H) and (g is None or g.shape == (B, T, H))
    assert k.dtype == v.dtype == torch.bfloat16, "the fused path is bf16-only"
    _capi.require_device(k, v, beta, g)
    for name, t in (("beta", beta), ("g", g)):
        _capi.require_f32(t, name)
    k, v, beta, g = (_capi.prep(t, n) for t, n in ((k, "k"), (v, "v"), (beta, "beta"), (g, "g")))
    w = torch.empty_like(k)
    u = torch.empty_like(v)
    status = _capi.load_library().thm_wy_fwd(
        _capi.ptr(k), _capi.ptr(v), _capi.ptr(beta), _capi.ptr(g), _capi.ptr(w), _capi.ptr(u),
        B, T, H, K, V, BT, _capi.THM_DTYPE[torch.bfloat16], int(sign), _capi.stream_of(k))
    _capi.check(status, "thm_wy_fwd")
    return w, u


def chunk_fwd_fused(q, k, w, u, g, scale: float, initial_state=None, output_final_state: bool = False,
                    save_new_value: bool = False):
    """o (and optionally v_new, final state) of chunk_fwd_h (delta form) followed
    by chunk_fwd_o, in one HIP kernel that never writes the per-chunk states
    (thm_chunk_gated_delta_fwd; bf16 q, k, w, u).  Returns (o, v_new or None, ht or None)."""
    B, T, H, K = k.shape
    V = u.shape[-1]
    assert T % BT == 0, f"T={T} must be a multiple of {BT}"
    assert q.shape == k.shape == w.shape and u.shape[:3] == (B, T, H) and (g is None or g.shape == (B, T, H))
    _check_state(initial_state, B, H, K, V)
    assert q.dtype == k.dtype == w.dtype == u.dtype == torch.bfloat16, "the fused path is bf16-only"
    _capi.require_device(q, k, w, u, g, initial_state)
    for name, t in (("g", g), ("initial_state", initial_state)):
        _capi.require_f32(t, name)
    q, k, w, u, g, h0 = (_capi.prep(t, n) for t, n in ((q, "q"), (k, "k"), (w, "w"), (u, "u"), (g, "g"),
                                                       (initial_state, "initial_state")))
    o = torch.empty_like(u)
    vn = torch.empty_like(u) if save_new_value else None
    ht = torch.empty(B, H, K, V, dtype=torch.float32, device=k.device) if output_final_state else None
    status = _capi.load_library().thm_chunk_gated_delta_fwd(
        _capi.ptr(q), _capi.ptr(k), _capi.ptr(w), _capi.ptr(u), _capi.ptr(g), _capi.ptr(h0), _capi.ptr(o),
        _capi.ptr(vn), _capi.ptr(ht), float(scale), B, T, H, K, V, BT, _capi.THM_DTYPE[torch.bfloat16],
        _capi.stream_of(k))
    _capi.check(status, "thm_chunk_gated_delta_fwd")
    return o, vn, ht


def chunk_fwd_fused_a(q, k, v, beta, A, g, scale: float, initial_state=None, output_final_state: bool = False,
                      save_new_value: bool = False):
    """The same as chunk_fwd_fused from the WY matrix A instead of w and u:
    v_new = A (beta (v - e^g k S)) = u - w S per chunk, in one HIP kernel
    (thm_chunk_gated_delta_fwd_a; bf16 q, k, v; fp32 beta, A, g).  Returns
    (o, v_new or None, ht or None)."""
    B, T, H, K = k.shape
    V = v.shape[-1]
    assert T % BT == 0, f"T={T} must be a multiple of {BT}"
    assert q.shape == k.shape and v.shape[:3] == (B, T, H) and beta.shape == (B, T, H)
    assert A.shape == (B, T, H, BT) and (g is None or g.shape == (B, T, H))
    _check_state(initial_state, B, H, K, V)
    assert q.dtype == k.dtype == v.dtype == torch.bfloat16, "the fused path is bf16-only"
    _capi.require_device(q, k, v, beta, A, g, initial_state)
    for name, t in (("beta", beta), ("A", A), ("g", g), ("initial_state", initial_state)):
        _capi.require_f32(t, name)
    q, k, v, beta, A, g, h0 = (_capi.prep(t, n) for t, n in ((q, "q"), (k, "k"), (v, "v"), (beta, "beta"),
                                                             (A, "A"), (g, "g"), (initial_state, "initial_state")))
    o = torch.empty_like(v)
    vn = torch.empty_like(v) if save_new_value else None
    ht = torch.empty(B, H, K, V, dtype=torch.float32, device=k.device) if output_final_state else None
    status = _capi.load_library().thm_chunk_gated_delta_fwd_a(
        _capi.ptr(q), _capi.ptr(k), _capi.ptr(v), _capi.ptr(beta), _capi.ptr(A), _capi.ptr(g), _capi.ptr(h0),
        _capi.ptr(o), _capi.ptr(vn), _capi.ptr(ht), float(scale), B, T, H, K, V, BT,
        _capi.THM_DTYPE[torch.bfloat16], _capi.stream_of(k))
    _capi.check(status, "thm_chunk_gated_delta_fwd_a")
    return o, vn, ht


def _fwd_records(q, k, v, beta, gate, gate_kind: int, scale: float, initial_state, output_final_state: bool):
    """The bf16 forward from (q, k, v, beta, gate) in one C call
    (thm_chunk_gated_delta_rule_fwd): (o, ht or None)."""
    fp = _capi.fastpath()
    if fp is not None:
        r = _capi.fast_result(fp.gated_delta_rule(q, k, v, beta, gate, gate_kind, initial_state, float(scale),
                                                  bool(output_final_state)), "thm_chunk_gated_delta_rule_fwd")
        if r is not None:
            return r
    B, T, H, K = k.shape
    V = v.shape[-1]
    assert T % BT == 0, f"T={T} must be a multiple of {BT}"
    assert q.shape == k.shape and v.shape[:3] == (B, T, H) and beta.shape == (B, T, H)
    assert gate is None or gate.shape == (B, T, H)
    _check_state(initial_state, B, H, K, V)
    assert q.dtype == k.dtype == v.dtype == torch.bfloat16, "the fused path is bf16-only"
    _capi.require_device(q, k, v, beta, gate, initial_state)
    for name, t in (("beta", beta), ("initial_state", initial_state)):
        _capi.require_f32(t, name)
    if gate_kind == _capi.THM_GATE_CUMULATIVE:
        _capi.require_f32(gate, "g")
    code = 0 if gate is None else _capi.dtype_code(gate, "a")
    q, k, v, beta, gate, h0 = (_capi.prep(t, n) for t, n in ((q, "q"), (k, "k"), (v, "v"), (beta, "beta"),
                                                            (gate, "gate"), (initial_state, "initial_state")))
    lib = _capi.load_library()
    nws = lib.thm_chunk_gated_delta_rule_workspace(B, T, H, K, V)
    ws = torch.empty(max(nws, 0), dtype=torch.uint8, device=k.device)
    o = torch.empty_like(v)
    ht = torch.empty(B, H, K, V, dtype=torch.float32, device=k.device) if output_final_state else None
    status = lib.thm_chunk_gated_delta_rule_fwd(
        _capi.ptr(q), _capi.ptr(k), _capi.ptr(v), _capi.ptr(beta), _capi.ptr(gate), _capi.ptr(h0), _capi.ptr(o),
        _capi.ptr(ht), _capi.ptr(ws), ws.numel(), float(scale), B, T, H, K, V, BT, _capi.THM_DTYPE[torch.bfloat16],
        code, gate_kind, _capi.stream_of(k))
    _capi.check(status, "thm_chunk_gated_delta_rule_fwd")
    return o, ht


def _gates_with_A(k, beta, a) -> bool:
    """Whether thm_wy_build_A_gates takes these; otherwise chunk_local_cumsum and
    build_A do, with their checks."""
    B, T, H, K = k.shape
    return (k.is_cuda and beta.device == k.device and a.device == k.device and k.dtype == beta.dtype == torch.float32
            and a.dtype in _capi.THM_DTYPE and T % BT == 0 and beta.shape == (B, T, H) and a.shape == (B, T, H))


def _build_A_gates(k, beta, a, logsigmoid: bool):
    """(A, g): build_A(k, beta, g) with g = chunk_local_cumsum(a), in one launch."""
    B, T, H, K = k.shape
    k, beta, a = (_capi.prep(t, n) for t, n in ((k, "k"), (beta, "beta"), (a, "a")))
    A = torch.empty(B, T, H, BT, dtype=torch.float32, device=k.device)
    g = torch.empty(B, T, H, dtype=torch.float32, device=k.device)
    status = _capi.load_library().thm_wy_build_A_gates(
        _capi.ptr(k), _capi.ptr(beta), _capi.ptr(a), _capi.ptr(A), _capi.ptr(g), B, T, H, K, BT,
        _capi.THM_DTYPE[k.dtype], _capi.THM_DTYPE[a.dtype],
        _capi.THM_GATE_LOGSIGMOID if logsigmoid else _capi.THM_GATE_IDENTITY, +1, _capi.stream_of(k))
    _capi.check(status, "thm_wy_build_A_gates")
    return A, g


def chunk_gated_delta_rule_fwd(q, k, v, beta, g, scale: float, initial_state=None,
                               output_final_state: bool = False, A: torch.Tensor | None = None,
                               return_intermediates: bool = False, a: torch.Tensor | None = None,
                               a_logsigmoid: bool = False, fused: bool | None = None,
                               fused_form: str = "A"):
    """o [B, T, H, V] (dtype of q) and the final state [B, H, K, V] fp32 (or None).

    bf16 inputs run fused kernels (``fused``, default for bf16 unless
    ``return_intermediates``, which needs w, u and the per-chunk states h):
    with ``fused_form`` "A" (default) one C call that forms per-chunk records
    (A and the gates) and runs recurrence and output from them, long sequences
    of few heads in segments side by side (w, u and the per-chunk states never
    formed), or chunk_fwd_fused_a when ``A`` is given; with "wy" wy_fwd (A and w, u in one kernel; unless ``A`` is given) and
    chunk_fwd_fused.  Otherwise build_A, recompute_w_u, chunk_fwd_h,
    chunk_fwd_o.
    ``g`` is the chunk-local cumulative log decay [B, T, H] fp32 (or None: no
    gate).  Alternatively pass the per-token log decay ``a`` (g = None): g is
    then formed on the GPU by chunk_local_cumsum(a), of log(sigmoid(a)) when
    ``a_logsigmoid``."""
    B, T, H, K = k.shape
    V = v.shape[-1]
    if a is not None:
        assert g is None, "pass either g or a"
    if fused is None:
        fused = k.dtype == torch.bfloat16 and not return_intermediates
    assert fused_form in ("A", "wy"), fused_form
    if fused and fused_form == "A" and A is None:
        if a is None:
            return _fwd_records(q, k, v, beta, g, _capi.THM_GATE_CUMULATIVE, scale, initial_state, output_final_state)
        kind = _capi.THM_GATE_LOGSIGMOID if a_logsigmoid else _capi.THM_GATE_IDENTITY
        return _fwd_records(q, k, v, beta, a, kind, scale, initial_state, output_final_state)
    if a is not None and A is None and not fused and _gates_with_A(k, beta, a):
        A, g = _build_A_gates(k, beta, a, a_logsigmoid)
    elif a is not None:
        g = chunk_local_cumsum(a, logsigmoid=a_logsigmoid)
    if fused and fused_form == "A":
        o, _, ht = chunk_fwd_fused_a(q, k, v, beta, A, g, scale, initial_state, output_final_state)
        return o, ht
    if fused and A is None:
        w, u = wy_fwd(k, v, beta, g, sign=+1)
    else:
        if A is None:
            A = build_A(k, beta, g)
        w, u = recompute_w_u.custom_kernel(recompute_w_u.Data(k=k, v=v, beta=beta, A=A, g=g,
                                                              B=B, T=T, H=H, K=K, V=V))
    if fused:
        o, _, ht = chunk_fwd_fused(q, k, w, u, g, scale, initial_state, output_final_state)
        return o, ht
    h, v_new, ht = chunk_fwd_h.custom_kernel(dict(k=k, w=w, u=u, g=g, initial_state=initial_state,
                                                  output_final_state=output_final_state))
    o = chunk_fwd_o.custom_kernel(dict(q=q, k=k, v=v_new, g=g, h=h, scale=scale))
    if return_intermediates:
        return o, ht, dict(A=A, g=g, w=w, u=u, h=h, v_new=v_new)
    return o, ht
