"""A row stride that spreads x over 2 GiB or more: no 32-bit offset reaches its last row, so a layer
quantized in groups of 32 runs the two-buffer GEMM (the one that addresses x in 64 bits), with every
epilogue and through the operators, as the same rows packed together would on that kernel."""

from __future__ import annotations

import pytest
import torch

import tokenforge.kernels.ops  # noqa: F401
from tests.numerics import cases
from tokenforge.kernels.config import SPAN_32BIT, default_config, m_bucket, untuned_config
from tokenforge.kernels.hip.w4a16 import w4a16_gemm_ex


def test_the_choice_follows_the_span_of_x() -> None:
    m, n, k, g = 160, 256, 256, 32
    base = default_config(m_bucket(m), n, k, g)
    assert (base.kernel, base.num_stages) == ("gemm_mfma", 2)
    assert untuned_config(m, n, k, g, SPAN_32BIT - 2) == untuned_config(m, n, k, g) != base
    assert untuned_config(m, n, k, g, SPAN_32BIT) == base


@pytest.mark.gpu
def test_rows_two_gib_apart(device: torch.device) -> None:
    m, n, k, g, stride = 160, 256, 256, 32, 1 << 23
    assert ((m - 1) * stride + k) * 2 >= SPAN_32BIT
    w = cases.on_device(cases.layer_weights(n, k, 0, g), device)
    packed = cases.activations(m, k, 0).to(device)
    x = torch.empty(m * stride, dtype=torch.float16, device=device).view(m, stride)[:, :k]
    x.copy_(packed)
    res = cases.activations(m, n, 1).to(device)
    args = (w.qweight_t, w.scales, w.qzeros, g, default_config(m_bucket(m), n, k, g), None)
    ops = torch.ops.tokenforge
    weights = (w.qweight_t, w.scales, w.qzeros, None)
    assert torch.equal(ops.w4a16_linear(x, *weights, g, "hip"), w4a16_gemm_ex(packed, *args))
    assert torch.equal(ops.w4a16_linear_residual(x, *weights, res, g, "hip"),
                       w4a16_gemm_ex(packed, *args, "residual", res))
    assert torch.equal(ops.w4a16_linear_silu_mul(x, *weights, g, "hip"), w4a16_gemm_ex(packed, *args, "silu_mul"))
