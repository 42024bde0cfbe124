"""GPU parity of the convolution where rows or segments are ragged: [B, D, S]
rows that start anywhere in a 16-byte vector or a 128-byte line (the last
row's end vector reaches past the tensor), and channels-last segments whose
last one overlaps the one before.  Against float64 (torch, CPU): fp32 sums of
W + 1 terms, W 2^-24 relative to the sum of the terms' magnitudes, and one
rounding to the output type; with SiLU also the hardware exponential's few
ulp.  The elements around the output are left alone."""
from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from theorem_amd.kernels import causal_conv1d

pytestmark = pytest.mark.gpu


def _reference(x, w, b, act):
    y = F.conv1d(F.pad(x.double().cpu(), (w.shape[1] - 1, 0)), w.double().cpu().unsqueeze(1), b.double().cpu(),
                 groups=x.shape[1])
    mag = F.conv1d(F.pad(x.double().cpu().abs(), (w.shape[1] - 1, 0)), w.double().cpu().abs().unsqueeze(1),
                   b.double().cpu().abs(), groups=x.shape[1])
    return (y * torch.sigmoid(y) if act else y), mag


def _check(out, x, w, b, act, what):
    ref, mag = _reference(x, w, b, act)
    bound = 16 * 2.0 ** -24 * mag + (2.0 ** -8 if x.dtype == torch.bfloat16 else 2.0 ** -23) * ref.abs()
    bad = (out.double().cpu() - ref).abs() > bound + 1e-30
    assert not bad.any(), f"{what}: {int(bad.sum())} elements beyond the bound"


def _inputs(B, D, S, W, dtype, dev):
    gen = torch.Generator().manual_seed(S * 8 + W)
    mk = lambda *n: torch.randn(*n, generator=gen).to(dtype).to(dev)  # noqa: E731
    return mk(B, D, S), mk(D, W), mk(D)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("S,W,act", [(65, 4, None), (63, 4, None), (127, 8, "silu"), (1021, 4, None), (1025, 3, "silu"),
                                     (2047, 4, "silu"), (2050, 5, None), (4099, 2, None), (131, 1, None)])
def test_ragged_rows(dev, dtype, S, W, act):
    B, D = 2, 7
    x, w, b = _inputs(B, D, S, W, dtype, dev)
    out = causal_conv1d.custom_kernel((x, w, b), activation=act)
    torch.cuda.synchronize()
    _check(out, x, w, b, act, f"S={S} W={W} {dtype}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ragged_rows_write_only_their_tensor(dev, dtype):
    # x and out inside larger buffers: NaN around x is not read into any
    # output, and what lies around out keeps its value.
    from theorem_amd.kernels import _capi

    D, S, W, pad = 5, 77, 4, 64
    x, w, b = _inputs(1, D, S, W, dtype, dev)
    xbuf = torch.full((2 * pad + D * S,), float("nan"), dtype=dtype, device=dev)
    obuf = torch.full_like(xbuf, 3.0)
    xbuf[pad:pad + D * S] = x.flatten()
    eb = x.element_size()
    st = _capi.load_library().thm_causal_conv1d_fwd(xbuf.data_ptr() + pad * eb, w.data_ptr(), b.data_ptr(),
                                                    obuf.data_ptr() + pad * eb, 1, D, S, W, _capi.THM_DTYPE[dtype],
                                                    _capi.THM_DTYPE[dtype], 0, _capi.stream_of(x))
    torch.cuda.synchronize()
    assert st == 0
    _check(obuf[pad:pad + D * S].reshape(1, D, S), x, w, b, None, "inside a buffer")
    assert (obuf[:pad] == 3.0).all() and (obuf[pad + D * S:] == 3.0).all()


# Where the rule sends rows from one form to another: 512 elements (scalar lanes
# up to there), bf16 rows that one wave of two groups holds (961 and, at any
# offset of its start, no longer), fp32 by width and by the size of the tensor
# (past and just within 256 MiB of x and out; few long rows).
@pytest.mark.parametrize("dtype,B,D,S,W,act", [
    (torch.bfloat16, 3, 5, 511, 4, "silu"), (torch.bfloat16, 3, 5, 513, 4, "silu"), (torch.bfloat16, 2, 40, 959, 3, None),
    (torch.bfloat16, 2, 40, 961, 4, None), (torch.bfloat16, 2, 40, 963, 8, "silu"), (torch.bfloat16, 1, 4100, 963, 4, None),
    (torch.bfloat16, 1, 4100, 1023, 4, "silu"), (torch.bfloat16, 1, 2050, 2049, 2, None),
    (torch.float32, 3, 5, 513, 6, "silu"), (torch.float32, 2, 40, 1021, 8, None), (torch.float32, 2, 40, 1025, 7, "silu"),
    (torch.float32, 2, 40, 2050, 5, None), (torch.float32, 4, 4096, 2049, 4, None), (torch.float32, 4, 4096, 2047, 4, None),
    (torch.float32, 1, 1030, 3003, 4, "silu"), (torch.float32, 1, 1025, 7001, 4, None), (torch.float32, 2, 40, 1601, 8, None)])
def test_ragged_rule(dev, dtype, B, D, S, W, act):
    x, w, b = _inputs(B, D, S, W, dtype, dev)
    out = causal_conv1d.custom_kernel((x, w, b), activation=act)
    torch.cuda.synchronize()
    if x.numel() > 1 << 22:  # the first and last channels of the first and last batch row
        n = x.shape[1]
        pick = torch.tensor([0, 1, 2, 3, n - 3, n - 2, n - 1], device=dev)
        out, x, w, b = out[[0, -1]][:, pick], x[[0, -1]][:, pick], w[pick], b[pick]
    _check(out, x, w, b, act, f"B={B} D={D} S={S} W={W} {dtype}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_ragged_vectors_write_only_their_tensor(dev, dtype):
    # As above with rows that take whole vectors in either type.
    from theorem_amd.kernels import _capi

    D, S, W, pad = 5, 1301, 8, 64
    x, w, b = _inputs(1, D, S, W, dtype, dev)
    xbuf = torch.full((2 * pad + D * S,), float("nan"), dtype=dtype, device=dev)
    obuf = torch.full_like(xbuf, 3.0)
    xbuf[pad:pad + D * S] = x.flatten()
    eb = x.element_size()
    st = _capi.load_library().thm_causal_conv1d_fwd(xbuf.data_ptr() + pad * eb, w.data_ptr(), b.data_ptr(),
                                                    obuf.data_ptr() + pad * eb, 1, D, S, W, _capi.THM_DTYPE[dtype],
                                                    _capi.THM_DTYPE[dtype], 0, _capi.stream_of(x))
    torch.cuda.synchronize()
    assert st == 0
    _check(obuf[pad:pad + D * S].reshape(1, D, S), x, w, b, None, "inside a buffer")
    assert (obuf[:pad] == 3.0).all() and (obuf[pad + D * S:] == 3.0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,S,D,W,act", [(1, 5, 64, 4, None), (2, 8, 64, 4, "silu"), (1, 15, 40, 3, None),
                                         (1, 17, 1048, 4, "silu"), (3, 33, 264, 8, None), (1, 64, 72, 1, None),
                                         (2, 131, 2056, 4, "silu"), (1, 1500, 16, 4, None), (8, 1100, 4096, 4, None)])
def test_channels_last_segments(dev, dtype, B, S, D, W, act):
    x, w, b = _inputs(B, D, S, W, dtype, dev)
    xc = x.transpose(1, 2).contiguous().transpose(1, 2)
    out = causal_conv1d.custom_kernel((xc, w, b), activation=act)
    torch.cuda.synchronize()
    assert out.stride() == xc.stride()
    if x.numel() > 1 << 22:  # the whole against the row kernel, its start against float64
        full = causal_conv1d.custom_kernel((x, w, b), activation=act)
        assert torch.equal(out, full)
        out, x = out[:1, :, :70], x[:1, :, :70]
    _check(out, x, w, b, act, f"B={B} S={S} D={D} W={W} {dtype}")
