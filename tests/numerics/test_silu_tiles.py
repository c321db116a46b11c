"""SiLU*mul applied in the epilogue of the LDS-tile GEMMs: every accumulator form (16x16 and 32x32
fragments, even and odd fragment counts per wave, the producer/consumer forms, fp8) at the edges of
its column mapping. A call equals torch's silu and multiply on the same config's plain output bit
for bit, also into rows whose stride is not a multiple of four (written value by value), and writes
nothing outside its outputs."""

from __future__ import annotations

import ctypes

import pytest
import torch

from tests.numerics import cases
from tokenforge.kernels import _lib
from tokenforge.kernels.config import GemmConfig
from tokenforge.kernels.hip._common import stream_of
from tokenforge.kernels.hip.w4a16 import to_c_config, w4a8_gemm_ex, w4a16_gemm

pytestmark = pytest.mark.gpu
G = 128
K = 256

CONFIGS = [
    GemmConfig("gemm_mfma", 256, 128, 64, 1, 8, 3),  # 32x32 fragments
    GemmConfig("gemm_mfma", 256, 192, 64, 1, 16, 3),  # ... sixteen waves
    GemmConfig("gemm_mfma", 256, 160, 64, 1, 8, 6),  # 16x16, five fragments a wave
    GemmConfig("gemm_mfma", 256, 224, 64, 1, 8, 6),  # ... seven, read one at a time
    GemmConfig("gemm_mfma", 256, 160, 64, 1, 8, 8),  # producer/consumer, odd and even counts
    GemmConfig("gemm_mfma", 128, 256, 64, 1, 8, 8),
    GemmConfig("gemm_fp8", 256, 160, 128, 1, 8, 3),
    GemmConfig("gemm_fp8", 256, 160, 128, 1, 8, 8),
    GemmConfig("gemm_fp8", 256, 128, 128, 1, 8, 8),
]


def _id(c: GemmConfig) -> str:
    return f"{c.kernel}-{c.block_m}x{c.block_n}-w{c.num_warps}-st{c.num_stages}"


@pytest.mark.parametrize("n", [16, 48, 320, 336, 640])  # N / 2 ends inside a fragment, a tile, a pair
@pytest.mark.parametrize("cfg", CONFIGS, ids=_id)
def test_silu_mul_in_the_tile_epilogue(cfg: GemmConfig, n: int, device: torch.device) -> None:
    w = cases.on_device(cases.layer_weights(n, K, 0), device)
    bias = cases.bias(n, 0).to(device)
    half = n // 2
    lib = _lib.lib()
    c = to_c_config(cfg)
    for m in (1, 17, cfg.block_m + 1):
        x = cases.activations(m, K, 0).to(device)
        xs = torch.rand((m, 1), device=device) + 0.5
        x8 = x.to(torch.float8_e4m3fn)
        fp8 = cfg.kernel == "gemm_fp8"
        if fp8:
            y = w4a8_gemm_ex(x8, xs.reshape(-1), w.qweight_t, w.scales, w.qzeros, G, cfg, bias)
        else:
            y = w4a16_gemm(x, w.qweight_t, w.scales, w.qzeros, G, cfg, bias)
        want = torch.nn.functional.silu(y[:, :half]) * y[:, half:]
        for ldo in (half, half + 3):
            buf = torch.full((m, ldo), 7.0, dtype=torch.float16, device=device)
            common = (w.qweight_t.data_ptr(), w.scales.data_ptr(), w.qzeros.data_ptr(), bias.data_ptr(), buf.data_ptr(),
                      ldo, m, n, K, G, ctypes.byref(c), _lib.EPILOGUE_SILU_MUL, None, 0, None, 0, stream_of(device))
            if fp8:
                rc = lib.tf_w4a8_linear_ex(x8.data_ptr(), K, xs.data_ptr(), 1, *common)
            else:
                rc = lib.tf_w4a16_linear_ex(x.data_ptr(), K, *common)
            _lib.check(rc, "linear")
            assert torch.equal(buf[:, :half], want), f"m={m} ldo={ldo}"
            assert bool((buf[:, half:] == 7.0).all()), f"m={m}: wrote past the outputs"
