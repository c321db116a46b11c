"""The K-split tile GEMM (waves split a tile's K, their sums meet in LDS) against an fp64 product on
the exact fp16 weights, at the edges of its tiles: M around its rows, N ending inside a tile and
inside a SiLU*mul column group (N / 16 odd), K shorter than a round of its waves and not a multiple
of it, K long enough that the pipelined loop goes round its ring more than twice and ends in every
position, every group size, K slices; fused epilogues equal torch's on its own plain output bit for
bit, and fewer rows per tile change no bit."""

from __future__ import annotations

from dataclasses import replace

import pytest
import torch

from tests.numerics import cases
from tokenforge.kernels import pack
from tokenforge.kernels.config import KSPLIT_TILES, GemmConfig, ksplit_config, ksplit_rows
from tokenforge.kernels.hip.w4a16 import w4a16_gemm_ex

pytestmark = pytest.mark.gpu

CONFIGS = [ksplit_config(mt, rt, wk) for mt, rt, wk in KSPLIT_TILES]


def _id(c: GemmConfig) -> str:
    return f"{c.block_m}x{c.block_n}-wk{c.waves_k}"


def _check(y: torch.Tensor, x: torch.Tensor, dense: torch.Tensor, want: torch.Tensor, what: str) -> None:
    """The numerics contract's bound (0.13 sqrt(K) eps max|x| max|w|) above half an fp16 ulp."""
    atol = 0.13 * x.shape[1] ** 0.5 * 2.0**-10 * float(x.abs().max()) * float(dense.abs().max())
    half_ulp = torch.ldexp(torch.ones_like(want), torch.frexp(want).exponent.clamp(min=-13) - 12)
    assert bool(((y.double() - want).abs() <= atol + half_ulp).all()), what


@pytest.mark.parametrize("n,k,g,split", [(16, 128, 128, 1), (208, 384, 32, 1), (352, 1152, 64, 1), (336, 2304, 128, 3)])
@pytest.mark.parametrize("cfg", CONFIGS, ids=_id)
def test_ksplit_tiles(cfg: GemmConfig, n: int, k: int, g: int, split: int, device: torch.device) -> None:
    cfg = replace(cfg, split_k=split)
    w = cases.on_device(cases.layer_weights(n, k, 0, g), device)
    dense = pack.dequantize_tf(w).double()
    bias = cases.bias(n, 0).to(device)
    half = n // 2
    for m in (1, cfg.block_m - 1, cfg.block_m + 1):
        x = cases.activations(m, k, 0).to(device)
        res = cases.activations(m, n, 1).to(device)
        args = (w.qweight_t, w.scales, w.qzeros, g, cfg, bias)
        y = w4a16_gemm_ex(x, *args)
        want = x.double() @ dense.t() + bias.double()
        _check(y, x, dense, want, f"m={m}")
        assert torch.equal(w4a16_gemm_ex(x, *args, "residual", res), res + y), f"residual m={m}"
        silu = torch.nn.functional.silu(y[:, :half]) * y[:, half:]
        assert torch.equal(w4a16_gemm_ex(x, *args, "silu_mul"), silu), f"silu_mul m={m}"
        fewer = ksplit_rows(cfg, m)
        assert torch.equal(w4a16_gemm_ex(x, w.qweight_t, w.scales, w.qzeros, g, fewer, bias), y), f"rows m={m}"


RING = 4  # the deepest weight ring of any tile, in rounds of a tile's waves along K


@pytest.mark.parametrize("cfg", CONFIGS, ids=_id)
def test_the_ring_comes_round(cfg: GemmConfig, device: torch.device) -> None:
    """K slices of 2 RING WK + 1 to 3 RING WK - 1 steps: the loop that counts its waits fills every ring
    slot at least twice and leaves 0 to RING - 1 rounds and a part of one to the tail."""
    n, m, g = 80, min(cfg.block_m + 1, 35), 64
    lengths = sorted({2 * RING * cfg.waves_k + 1, 2 * RING * cfg.waves_k + cfg.waves_k,
                      (2 * RING + 1) * cfg.waves_k + 1, (2 * RING + 2) * cfg.waves_k + 1, 3 * RING * cfg.waves_k - 1})
    for steps, split in [(s, 1) for s in lengths] + [(3 * lengths[0], 3)]:
        k = 128 * steps
        w = cases.on_device(cases.layer_weights(n, k, 0, g), device)
        dense = pack.dequantize_tf(w).double()
        x = cases.activations(m, k, 0).to(device)
        args = (x, w.qweight_t, w.scales, w.qzeros, g, replace(cfg, split_k=split), None)
        y = w4a16_gemm_ex(*args)
        _check(y, x, dense, x.double() @ dense.t(), f"{steps} steps, split {split}")
        silu = torch.nn.functional.silu(y[:, : n // 2]) * y[:, n // 2 :]
        assert torch.equal(w4a16_gemm_ex(*args, "silu_mul"), silu), f"silu_mul, {steps} steps, split {split}"
