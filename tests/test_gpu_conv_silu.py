"""SiLU of bf16 outputs holds what the fp32 path holds before the rounding: with
x = 1, W = 1 and fp32 weights both types see the same accumulators, so the bf16
output is the fp32 output rounded, bit for bit, in every convolution kernel and
at the edges of the exponential's range (infinities and NaN among them)."""
from __future__ import annotations

import pytest
import torch

from theorem_amd.kernels import causal_conv1d

pytestmark = pytest.mark.gpu
D = 1 << 18


def _weights(dev):
    gen = torch.Generator().manual_seed(0)
    w = torch.randn(D, generator=gen) * 4
    w[: D // 4] *= 40 * torch.rand(D // 4, generator=gen)  # past |v| = 80, where the quotient leaves the normal range
    edge = torch.tensor([0.0, -0.0, 79.999, 80.0, -79.999, -80.0, -87.0, -87.33, -87.34, -88.0, -88.7, -88.73, -89.0, 88.7,
                         -103.0, 3e38, -3e38, float("inf"), float("-inf"), float("nan"), 1e-30, -1e-30])
    w[1000::1000][: len(edge)] = edge  # alone among ordinary channels, and side by side
    w[-len(edge):] = edge
    return w.reshape(D, 1).to(dev)


def _call(form, w, dtype):
    dev = w.device
    if form == "rows":
        return causal_conv1d.custom_kernel((torch.ones(1, D, 64, dtype=dtype, device=dev), w, None), activation="silu")
    if form == "ragged rows":
        return causal_conv1d.custom_kernel((torch.ones(1, D, 77, dtype=dtype, device=dev), w, None), activation="silu")
    if form == "channels-last":
        x = torch.ones(1, 40, D, dtype=dtype, device=dev).transpose(1, 2)
        return causal_conv1d.custom_kernel((x, w, None), activation="silu")
    L = 1 if form == "step" else 2
    x, state = torch.ones(1, D, L, dtype=dtype, device=dev), torch.ones(1, D, 1, dtype=dtype, device=dev)
    return causal_conv1d.causal_conv1d_update(x, state, w, None, activation="silu")


@pytest.mark.parametrize("form", ["rows", "ragged rows", "channels-last", "step", "update"])
def test_bf16_is_fp32_rounded(dev, form):
    w = _weights(dev)
    got, full = (_call(form, w, dt) for dt in (torch.bfloat16, torch.float32))
    want = full.bfloat16()
    bits = (got.view(torch.int16) == want.view(torch.int16)) | (got.isnan() & want.isnan())
    assert bits.all(), f"{form}: {int((~bits).sum())} of {bits.numel()} differ"
