"""The workloads whose time this framework is judged by: what a user's program has it do, through its public
entry points, from one decode step to a batch of long sequences.

A case is a dict of plain values.  Fields: ``op``; for the convolution B, D, S, W, ``dtype``, ``act`` (SiLU);
for the Gated DeltaNet ops B, T, H, K, V, ``dtype`` and, for the whole forward, ``state`` (it continues from a
given state).  The ops:

  conv      causal_conv1d.custom_kernel on x [B, D, S] contiguous: the prefill of a Mamba-2 style block.
  conv_cl   the same on a channels-last x (a [B, D, S] view of [B, S, D]), the layout such a block holds its
            activations in.
  update    causal_conv1d.causal_conv1d_update: one decode step of one token per sequence.
  wu        recompute_w_u.custom_kernel.
  h_ref     chunk_fwd_h.custom_kernel, the reference's form (k, v, g -> h).
  h         chunk_fwd_h.custom_kernel, delta form (h, v_new and the final state).
  o         chunk_fwd_o.custom_kernel.
  chain     chain.chunk_gated_delta_rule_fwd from (q, k, v, beta, a): prefill of a Gated DeltaNet layer,
            with the state handed to the decode that follows.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

from theorem_amd import chain
from theorem_amd.kernels import causal_conv1d, chunk_fwd_h, chunk_fwd_o, recompute_w_u

BT = 64
_DT = {"bf16": torch.bfloat16, "f32": torch.float32}
_CONV = ("conv", "conv_cl", "update")
# No drawn case is larger than chain_batch below: B T H token-heads, conv elements.
_MAX_TOKENS = {"bf16": 1 << 20, "f32": 1 << 18}
_MAX_CONV = 1 << 27


def listed():
    return [
        # One token for each of 64 sequences being decoded, between other layers' kernels: launch and latency.
        dict(name="conv_update", op="update", B=64, D=4096, S=1, W=4, dtype="bf16", act=True),
        # The reference's largest convolution benchmark shape, fp32 and without an activation as there.
        dict(name="conv_task_f32", op="conv", B=1, D=2560, S=4096, W=4, dtype="f32", act=False),
        # Prompts of a length that is no multiple of anything, bf16 with the block's SiLU.
        dict(name="conv_ragged", op="conv", B=4, D=4096, S=4003, W=4, dtype="bf16", act=True),
        # The same from a block that keeps its activations channels-last; the convolved width of such a
        # block is its inner width and two state groups.
        dict(name="conv_cl", op="conv_cl", B=2, D=4352, S=5001, W=4, dtype="bf16", act=True),
        # The reference's largest benchmark shapes of these two ops, fp32 as there: small calls.
        dict(name="wu_task_f32", op="wu", B=2, T=1024, H=3, K=64, V=64, dtype="f32"),
        dict(name="h_task_f32", op="h_ref", B=2, T=1024, H=3, K=64, V=64, dtype="f32"),
        # The state recurrence alone over one long sequence, with every output a later pass needs.
        dict(name="h_long", op="h", B=1, T=8192, H=16, K=128, V=128, dtype="bf16"),
        # The output stage alone at an ordinary batch.
        dict(name="o_batch", op="o", B=4, T=2048, H=16, K=128, V=128, dtype="bf16"),
        # Prefill of one short prompt: a few launches, little work in each.
        dict(name="chain_short", op="chain", B=1, T=192, H=16, K=128, V=128, dtype="bf16", state=False),
        # Prefill of one long prompt, continued from an earlier piece's state: the usual serving call.
        dict(name="chain_prompt", op="chain", B=1, T=8192, H=16, K=128, V=128, dtype="bf16", state=True),
        # A batch of long sequences (the benchmark's largest size): training's forward, offline prefill.
        dict(name="chain_batch", op="chain", B=8, T=8192, H=16, K=128, V=128, dtype="bf16", state=False),
        # The whole forward in the reference's own precision.
        dict(name="chain_f32", op="chain", B=2, T=2048, H=8, K=128, V=128, dtype="f32", state=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["conv", "conv_cl", "update", "wu", "h_ref", "h", "o", "chain", "chain", "chain"])
    dtype = rng.choice(["bf16", "bf16", "f32"])
    if op in _CONV:
        # Widths of real blocks are multiples of 8 or 64; lengths are whatever the prompt has.
        while True:
            B = _log_int(rng, 1, 128) if op == "update" else _log_int(rng, 1, 8)
            D = 8 * _log_int(rng, 8, 768)
            S = 1 if op == "update" else _log_int(rng, 64, 8192)
            if B * D * S <= _MAX_CONV:
                return dict(op=op, B=B, D=D, S=S, W=rng.choice([2, 3, 4, 4, 4]), dtype=dtype,
                            act=rng.random() < 0.6)
    while True:
        B, T, H = _log_int(rng, 1, 8), BT * _log_int(rng, 1, 128), _log_int(rng, 1, 32)
        if B * T * H <= _MAX_TOKENS[dtype]:
            break
    c = dict(op=op, B=B, T=T, H=H, K=rng.choice([64, 128]), V=rng.choice([64, 128]), dtype=dtype)
    if op == "chain":
        c["state"] = rng.random() < 0.5
    return c


# ----------------------------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda")


def _log_decay(gen, B, T, H):
    """Per-token log decay of a gated layer: one rate per head, over the logarithm from a memory of hundreds
    of tokens to one of a token or two, and a factor that varies from token to token."""
    rate = torch.exp(torch.empty(H, device="cuda").uniform_(math.log(0.002), math.log(0.8), generator=gen))
    return -rate * (0.5 + torch.rand(B, T, H, generator=gen, device="cuda"))


def _cumsum(a):
    B, T, H = a.shape
    return a.reshape(B, T // BT, BT, H).cumsum(dim=2).reshape(B, T, H)


def _chunked(x):
    """[B, T, H, D] -> [B, T/64, H, 64, D] in float64."""
    B, T, H, D = x.shape
    return x.double().reshape(B, T // BT, BT, H, D).transpose(2, 3).contiguous()


def _unchunk(x):
    B, NT, H, _, D = x.shape
    return x.transpose(2, 3).reshape(B, NT * BT, H, D)


def _t(x):
    return x.transpose(-1, -2).contiguous()


def _wy_matrix(kc, bc, gc):
    """(I + M)^{-1} in float64, M = strict_lower(beta_i (k_i . k_j) e^{g_i - g_j}): M^64 = 0, so the product
    (I - M)(I + M^2)(I + M^4) ... (I + M^32) is the inverse."""
    M = torch.tril((kc @ _t(kc)) * bc * torch.exp((gc - gc.transpose(-1, -2)).clamp_max(0.0)), diagonal=-1)
    eye = torch.eye(BT, dtype=torch.float64, device=kc.device)
    X, P = eye - M, M @ M
    for i in range(5):
        X = X @ (eye + P)
        if i < 4:
            P = P @ P
    return X


def _inputs(case, seed):
    gen = _gen(seed)
    dt = _DT[case["dtype"]]
    op = case["op"]
    if op in _CONV:
        B, D, S, W = (case[n] for n in "BDSW")
        if op == "conv_cl":
            x = _randn(gen, B, S, D).to(dt).transpose(1, 2)
        elif op == "update":
            x = _randn(gen, B, D).to(dt)
        else:
            x = _randn(gen, B, D, S).to(dt)
        d = dict(x=x, weight=(_randn(gen, D, W) / 2).to(dt), bias=(_randn(gen, D) * 0.1).to(dt))
        if op == "update":
            d["conv_state"] = _randn(gen, B, D, W).to(dt)
        return d
    B, T, H, K, V = (case[n] for n in "BTHKV")
    k = F.normalize(_randn(gen, B, T, H, K), dim=-1).to(dt)
    a = _log_decay(gen, B, T, H)
    if op == "h_ref":
        return dict(k=k, v=_randn(gen, B, T, H, V).to(dt), g=_cumsum(a))
    if op == "o":
        return dict(q=F.normalize(_randn(gen, B, T, H, K), dim=-1).to(dt), k=k, v=_randn(gen, B, T, H, V).to(dt),
                    g=_cumsum(a), h=_randn(gen, B, T // BT, H, K, V) * 0.1)
    v = _randn(gen, B, T, H, V).to(dt)
    beta = torch.sigmoid(_randn(gen, B, T, H))
    if op == "chain":
        h0 = _randn(gen, B, H, K, V) * 0.1 if case["state"] else None
        return dict(q=F.normalize(_randn(gen, B, T, H, K), dim=-1).to(dt), k=k, v=v, beta=beta, a=a, h0=h0)
    g = _cumsum(a)
    kc, bc, gc = _chunked(k), _chunked(beta.unsqueeze(-1)), _chunked(g.unsqueeze(-1))
    A = _wy_matrix(kc, bc, gc)
    if op == "wu":
        return dict(k=k, v=v, beta=beta, g=g, A=_unchunk(A).float().contiguous())
    w = _unchunk(A @ (kc * bc * torch.exp(gc))).to(dt).contiguous()
    u = _unchunk(A @ (_chunked(v) * bc)).to(dt).contiguous()
    return dict(k=k, w=w, u=u, g=g)


def prepare(case, seed):
    d = _inputs(case, seed)
    op = case["op"]
    act = "silu" if case.get("act") else None
    if op in ("conv", "conv_cl"):
        return dict(op=op, data=(d["x"], d["weight"], d["bias"]), act=act)
    if op == "update":
        return dict(op=op, act=act, **d)
    B, T, H, K, V = (case[n] for n in "BTHKV")
    if op == "wu":
        return dict(op=op, data=recompute_w_u.Data(**d, B=B, T=T, H=H, K=K, V=V))
    if op == "h":
        d["output_final_state"] = True
    if op == "o":
        d["scale"] = K ** -0.5
    if op == "chain":
        d["scale"] = K ** -0.5
    return dict(op=op, data=d)


# ----------------------------------------------------------------------------------------------- one pass

def run(state):
    op = state["op"]
    if op in ("conv", "conv_cl"):
        return causal_conv1d.custom_kernel(state["data"], activation=state["act"])
    if op == "update":
        out = causal_conv1d.causal_conv1d_update(state["x"], state["conv_state"], state["weight"], state["bias"],
                                                 activation=state["act"])
        return out, state["conv_state"]
    d = state["data"]
    if op == "wu":
        return recompute_w_u.custom_kernel(d)
    if op in ("h", "h_ref"):
        return chunk_fwd_h.custom_kernel(d)
    if op == "o":
        return chunk_fwd_o.custom_kernel(d)
    return chain.chunk_gated_delta_rule_fwd(d["q"], d["k"], d["v"], d["beta"], None, d["scale"],
                                            initial_state=d["h0"], output_final_state=True, a=d["a"])


# ----------------------------------------------------------------------------------------------- what it takes

def work(case):
    """Each input read once, each output written once; products of whole 64-token chunks, those with a
    triangular matrix at half."""
    eb = 2 if case["dtype"] == "bf16" else 4
    op = case["op"]
    if op in _CONV:
        B, D, S, W = (case[n] for n in "BDSW")
        n = B * D * S
        byt = 2 * n * eb + D * (W + 1) * eb
        if op == "update":
            byt += 2 * B * D * W * eb
        return {"bytes": byt, "flops": 2 * n * W}
    B, T, H, K, V = (case[n] for n in "BTHKV")
    N, NC = B * T * H, B * (T // BT) * H
    if op == "wu":
        return {"bytes": N * (2 * (K + V) * eb + 8 + 4 * BT), "flops": N * BT * (K + V)}
    if op == "h_ref":
        return {"bytes": N * ((K + V) * eb + 4) + NC * K * V * 4, "flops": 2 * N * K * V}
    if op == "h":
        return {"bytes": N * ((2 * K + 2 * V) * eb + 4) + (NC + B * H) * K * V * 4, "flops": 4 * N * K * V}
    if op == "o":
        return {"bytes": N * ((2 * K + 2 * V) * eb + 4) + NC * K * V * 4, "flops": N * (2 * K * V + BT * (K + V))}
    states = (2 if case["state"] else 1) * B * H * K * V * 4
    # k k^T, the inverse, A (v - k S) with k S, q k^T, its product with v_new, q S, k^T v_new.
    flops = N * (BT * K + BT * BT // 3 + BT * V + 2 * K * V + BT * K + BT * V + 2 * K * V + 2 * K * V)
    return {"bytes": N * ((2 * K + 2 * V) * eb + 8) + states, "flops": flops}


def tolerance(case):
    """About four times the error against 64 bits that the ops show at these sizes: the rounding of outputs,
    probabilities and states to bf16, or of sums in fp32 (the fp32 products run as three bf16 products)."""
    bf16 = case["dtype"] == "bf16"
    if case["op"] in _CONV:
        return {"rel": 7e-3 if bf16 else 4e-7}
    return {"rel": 1.5e-2 if bf16 else 4e-5}


# ----------------------------------------------------------------------------------------------- in 64 bits

def _exact_conv(case, d):
    W = case["W"]
    x, w, b = d["x"], d["weight"].double(), d["bias"].double()

    def act(y):
        return y * torch.sigmoid(y) if case["act"] else y

    if case["op"] == "update":
        win = torch.cat([d["conv_state"].double(), x.double().unsqueeze(-1)], dim=-1)
        out = act(b + (win[..., -W:] * w).sum(dim=-1))
        return out, win[..., 1:].to(d["conv_state"].dtype)
    outs = []
    for xb in x:  # one batch row at a time
        xp = F.pad(xb.double(), (W - 1, 0))
        acc = b[:, None].expand(xb.shape).clone()
        for i in range(W):
            acc += w[:, i:i + 1] * xp[:, i:i + xb.shape[1]]
        outs.append(act(acc))
    return torch.stack(outs)


def _recurrence(kc, gc, vc, wc=None, S=None, after=False):
    """States per chunk (before it, or after it with ``after``), v_new and the last state, in float64."""
    B, NT, H, _, K = kc.shape
    V = vc.shape[-1]
    S = torch.zeros(B, H, K, V, dtype=torch.float64, device=kc.device) if S is None else S.double()
    hs = torch.empty(B, NT, H, K, V, dtype=torch.float64, device=kc.device)
    vn = torch.empty_like(vc)
    for c in range(NT):
        if not after:
            hs[:, c] = S
        vn[:, c] = vc[:, c] if wc is None else vc[:, c] - wc[:, c] @ S
        gl = gc[:, c, :, -1:]
        S = torch.exp(gl) * S + _t(kc[:, c]) @ (vn[:, c] * torch.exp(gl - gc[:, c]))
        if after:
            hs[:, c] = S
    return hs, vn, S


def _outputs(qc, kc, gc, vn, hs, scale):
    out = torch.empty_like(vn)
    for c in range(qc.shape[1]):  # one chunk of every sequence at a time
        P = torch.tril((qc[:, c] @ _t(kc[:, c])) * torch.exp((gc[:, c] - gc[:, c].transpose(-1, -2)).clamp_max(0.0)))
        out[:, c] = scale * (P @ vn[:, c] + torch.exp(gc[:, c]) * (qc[:, c] @ hs[:, c]))
    return out


def exact(case, seed):
    d = _inputs(case, seed)
    op = case["op"]
    if op in _CONV:
        return _exact_conv(case, d)
    kc = _chunked(d["k"])
    if op == "chain":
        gc = _chunked(_cumsum(d["a"].double()).unsqueeze(-1))
        bc = _chunked(d["beta"].unsqueeze(-1))
        A = _wy_matrix(kc, bc, gc)
        wc, uc = A @ (kc * bc * torch.exp(gc)), A @ (_chunked(d["v"]) * bc)
        hs, vn, S = _recurrence(kc, gc, uc, wc, d["h0"])
        return _unchunk(_outputs(_chunked(d["q"]), kc, gc, vn, hs, case["K"] ** -0.5)), S
    gc = _chunked(d["g"].unsqueeze(-1))
    if op == "wu":
        A, bc = _chunked(d["A"]), _chunked(d["beta"].unsqueeze(-1))
        return _unchunk(A @ (kc * bc * torch.exp(gc))), _unchunk(A @ (_chunked(d["v"]) * bc))
    if op == "h_ref":
        return _recurrence(kc, gc, _chunked(d["v"]), after=True)[0]
    if op == "h":
        hs, vn, S = _recurrence(kc, gc, _chunked(d["u"]), _chunked(d["w"]))
        return hs, _unchunk(vn), S
    return _unchunk(_outputs(_chunked(d["q"]), kc, gc, _chunked(d["v"]), d["h"].double(), case["K"] ** -0.5))
