"""``pack_awq`` (one kernel from the AWQ format to the tile layout) against the oracle's two layout
steps, bit for bit, where its 256-row x 256-K blocks end: narrow last tiles, K chunks short of a
128-wide step, every group size, and scales that allow no 16-byte access."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import pack as opack
from tokenforge.kernels import pack

pytestmark = pytest.mark.gpu

SHAPES = [(n, k, g) for n in (8, 16, 24, 200, 256, 264, 528) for k, g in ((32, 32), (96, 32), (256, 32), (288, 32), (64, 64),
                                                                         (320, 64), (128, 128), (384, 128))]


@pytest.mark.parametrize("n,k,g", SHAPES)
def test_pack_awq_equals_the_oracle(n: int, k: int, g: int, device: torch.device) -> None:
    rng = np.random.default_rng(n * 1000 + k + g)
    qweight = rng.integers(-(2**31), 2**31, (k, n // 8), dtype=np.int64).astype(np.int32)
    qzeros = rng.integers(-(2**31), 2**31, (k // g, n // 8), dtype=np.int64).astype(np.int32)
    scales = rng.uniform(1e-3, 1e-2, (k // g, n)).astype(np.float16)
    want = opack.pack_awq_tiles(qweight, qzeros, scales, g)
    qw, qz = torch.from_numpy(qweight).to(device), torch.from_numpy(qzeros).to(device)
    aligned = torch.from_numpy(scales).to(device)
    shifted = torch.empty(scales.size + 1, dtype=torch.float16, device=device)[1:].view(scales.shape)
    shifted.copy_(aligned)
    for sc in (aligned, shifted):
        got = pack.pack_awq(qw, qz, sc, g)
        assert np.array_equal(got.qweight_t.cpu().numpy(), want.qweight_t)
        assert np.array_equal(got.scales.cpu().numpy().view(np.uint16), want.scales.view(np.uint16))
        assert np.array_equal(got.qzeros.cpu().numpy(), want.qzeros)
