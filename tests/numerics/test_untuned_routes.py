"""``w4a16_linear`` on layers nobody has tuned, on both sides of every line of the launch choice: the
library takes the chosen config for the shape, and the result is within the numerics contract's bound
of an fp64 product on the exact fp16 weights."""

from __future__ import annotations

import pytest
import torch

import tokenforge.kernels.ops  # noqa: F401
from tests.numerics import cases
from tokenforge.kernels import pack

SMALL_M = (1, 2, 4, 5, 8, 9, 17)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(("n", "k", "g", "ms"), [
    (512, 1024, 128, SMALL_M), (512, 1152, 64, SMALL_M), (512, 2176, 32, SMALL_M), (520, 1024, 64, SMALL_M),
    (512, 7296, 64, SMALL_M), (8224, 4224, 128, SMALL_M), (8208, 8320, 128, SMALL_M), (4096, 512, 128, SMALL_M), (4112, 4224, 128, SMALL_M), (4112, 8320, 64, SMALL_M), (10240, 384, 128, SMALL_M),
    (10256, 1280, 32, SMALL_M), (10240, 4096, 128, SMALL_M), (256, 12544, 128, SMALL_M), (3600, 640, 128, (129, 1025)),
    (264, 320, 64, (129, 300, 1025)), (272, 384, 32, (129, 1025)), (3848, 256, 64, (3585,)),
])
def test_untuned_layers(n: int, k: int, g: int, ms: tuple[int, ...], device: torch.device) -> None:
    qw, qz, sc = (torch.from_numpy(a).to(device) for a in cases.baseline_layer(n, k, 0, g))
    w = pack.pack_awq(qw, qz, sc, g)
    dense = pack.dequantize_tf(w).double()
    for m in ms:
        x = cases.activations(m, k, 0).to(device)
        y = torch.ops.tokenforge.w4a16_linear(x, w.qweight_t, w.scales, w.qzeros, None, g, "hip")
        want = x.double() @ dense.t()
        # the contract's bound (0.13 sqrt(K) eps max|x| max|w|) above half an fp16 ulp of the output
        atol = 0.13 * k**0.5 * 2.0**-10 * float(x.abs().max()) * float(dense.abs().max())
        half_ulp = torch.ldexp(torch.ones_like(want), torch.frexp(want).exponent.clamp(min=-13) - 12)
        assert bool(((y.double() - want).abs() <= atol + half_ulp).all()), f"m={m}"
