"""``w4a8_linear`` on both sides of the rules that pick the kernel for 9 to 17 rows (the GEMV that
decodes while staging, or the conversion and the K-split tile): with a unit scale the operator equals
the W4A16 kernel of the same config on the decoded x bit for bit, and row scales that are powers of
two scale its rows exactly."""

from __future__ import annotations

import pytest
import torch

from tests.numerics import cases
from tests.numerics.test_w4a8 import _codes
from tokenforge.kernels import ops
from tokenforge.kernels.hip.w4a16 import w4a16_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("n", "k", "g"), [(896, 896, 64), (512, 1536, 32), (1040, 4096, 128), (4112, 2048, 128),
                                           (528, 4224, 128)])
@pytest.mark.parametrize("m", [9, 16, 17])
def test_rows_9_to_17(m: int, n: int, k: int, g: int, device: torch.device) -> None:
    w = cases.on_device(cases.layer_weights(n, k, 0, g), device)
    x8 = _codes(m, k, m).to(device).view(torch.float8_e4m3fn)
    x16 = x8.to(torch.float16)
    weights = (w.qweight_t, w.scales, w.qzeros)
    dev = torch.device("cuda", torch.cuda.current_device())
    cfg = ops._w4a8_config(ops._gpu_config(dev, m, n, k, g), m, n, k, g)
    one = torch.ones(1, dtype=torch.float32, device=device)
    y = torch.ops.tokenforge.w4a8_linear(x8, one, *weights, None, g, "hip")
    assert torch.equal(y, w4a16_gemm(x16, *weights, g, cfg))
    # Powers of two as row scales move no rounding: the scaled result is the plain one, scaled.
    s = 2.0 ** torch.arange(-4, m - 4, device=device).clamp(max=0).float().reshape(m, 1)
    y = y.float() * s
    got = torch.ops.tokenforge.w4a8_linear(x8, s, *weights, None, g, "hip").float()
    normal = y.abs() >= 2.0**-14  # below that fp16 rounds at another place
    assert torch.equal(got[normal], y[normal])
