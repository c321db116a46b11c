"""The launch choice for layers nobody has tuned, on the CPU: every (shape, M, group size) gets a
config that the library has compiled, allows for the group size and whose kernel serves the shape
(its N, K and M conditions, restated here), the same one whatever the epilogue; and a tuned K-split
tile keeps its columns and K split when it loses spare rows."""

from __future__ import annotations

import ctypes

import pytest

from tokenforge.kernels import _lib
from tokenforge.kernels.config import (
    KSPLIT_TILES,
    default_config,
    ksplit_config,
    ksplit_rows,
    m_bucket,
    tuned_at,
    untuned_config,
)
from tokenforge.kernels.hip.w4a16 import to_c_config

SHAPES = [(8, 128), (16, 256), (200, 256), (1000, 1024), (1152, 896), (896, 4864), (2544, 256), (13448, 768), (37888, 3584),
          (3584, 18944), (4608, 3584), (11040, 5504), (608, 64), (256, 96)]


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize(("n", "k"), SHAPES)
def test_untuned_configs_run_their_shape(n: int, k: int, group: int) -> None:
    if k % group:
        pytest.skip("not a layer")
    for m in (1, 2, 4, 5, 8, 9, 16, 17, 33, 100, 129, 333, 1000, 4096, 5000):
        cfg = untuned_config(m, n, k, group)
        cfg.validate(group)
        # without rows the library checks the sizes and the config and returns
        c = to_c_config(cfg)
        rc = _lib.lib().tf_w4a16_linear_ex(None, k, None, None, None, None, None, n, 0, n, k, group, ctypes.byref(c), 0,
                                           None, 0, None, 0, None)
        assert rc == 0, f"m={m}: {cfg}"
        if cfg.ksplit:
            assert n % 16 == 0 and k % 128 == 0
            assert cfg.split_k <= k // 128
        elif cfg.stream:
            assert m <= cfg.block_m and n % 32 == 0 and k // 128 >= cfg.num_warps
        elif cfg.kernel == "gemm_mfma" and cfg.block_k == 64:
            assert group >= 64 or cfg.num_stages == 2
            assert cfg.split_k <= k // 64
        else:
            assert cfg.family == "gemv" or m >= 9


def test_rows_of_a_tuned_tile_follow_m() -> None:
    tuned = ksplit_config(4, 5, 4)
    assert [ksplit_rows(tuned, m).block_m for m in (1, 16, 33, 48, 49, 64, 65, 90, 100, 128)] == [
        16, 16, 48, 48, 64, 64, 48, 48, 64, 64]
    for mt, rt, wk in KSPLIT_TILES:
        cfg = ksplit_config(mt, rt, wk, 2)
        for m in (1, 16, 40, 77, 300):
            got = ksplit_rows(cfg, m)
            assert (got.block_n, got.waves_k, got.split_k) == (cfg.block_n, cfg.waves_k, cfg.split_k)
            assert -(-m // got.block_m) == -(-m // cfg.block_m)


def test_layers_outside_the_model_keep_the_bucket_default() -> None:
    for m in (1, 8, 100):
        assert untuned_config(m, 200, 1024, 128) == default_config(m_bucket(m), 200, 1024, 128)
    assert untuned_config(64, 1 << 20, 1 << 13, 128) == default_config(64, 1 << 20, 1 << 13, 128)
    # ... 4 GiB of weights, which the library refuses at this M: the form's offsets are 32-bit


def test_a_tuned_tile_gives_way_inside_its_bucket_only() -> None:
    gate_up = (37888, 3584, 128)
    tuned64, tuned128 = ksplit_config(4, 3, 2), ksplit_config(4, 5, 4)
    for m in range(49, 65):  # the model's rows are the bucket's: the tuner measured these tiles
        assert tuned_at(tuned64, m, *gate_up) == tuned64
    assert tuned_at(tuned128, 80, *gate_up) == ksplit_config(5, 3, 2)  # one tile of 80 rows against two of 48
    for m in (9, 33, 65, 80, 100, 127):  # a choice of the caller's own tuner only loses spare rows
        for cfg in (tuned64, tuned128):
            assert tuned_at(cfg, m, *gate_up, own=True) == ksplit_rows(cfg, m)


def test_tuned_choices_fit_their_layer() -> None:
    for n, k in ((37888, 3584), (4608, 3584), (3584, 3584), (3584, 18944), (256, 1024)):
        for mt, rt, wk in KSPLIT_TILES:
            for m in (9, 20, 40, 70, 100, 129, 200, 300, 500):
                for split in (1, 4):
                    cfg = tuned_at(ksplit_config(mt, rt, wk, split), m, n, k, 128)
                    cfg.validate(128)
                    assert not cfg.ksplit or (n % 16 == 0 and k % 128 == 0)
                    assert cfg.split_k <= k // 64


@pytest.mark.parametrize(("n", "k", "m", "kernel"), [
    (4096, 1024, 3, (16, 4)), (4096, 2048, 3, (16, 8)), (4096, 2944, 3, "base"), (5120, 11008, 2, "base"),
    (4096, 2048, 2, (16, 4)), (8192, 4096, 2, (16, 8)), (4096, 11008, 4, (16, 16)), (4096, 5632, 2, (16, 16)),
    (8192, 8192, 4, "base"), (4608, 4096, 1, "base"), (528, 4096, 3, (16, 8)), (3584, 18944, 3, (16, 16)),
    (4608, 18944, 3, "base"), (6160, 8192, 3, (16, 8)), (16400, 4096, 3, "base"), (17712, 256, 6, (16, 2)),
    (31200, 1408, 17, "base"), (6144, 13696, 11, "base"), (31824, 256, 16, "base"),
])
def test_decode_rows_keep_the_default_where_it_is_faster(n: int, k: int, m: int, kernel: object) -> None:
    cfg = untuned_config(m, n, k, 128)
    if kernel == "base":
        assert cfg == default_config(m_bucket(m), n, k, 128)
    else:
        assert (cfg.kernel, cfg.block_k, (cfg.block_n, cfg.num_warps)) == ("gemv_mfma", 128, kernel)


@pytest.mark.parametrize(("n", "k", "m", "tile"), [
    (4096, 4096, 3584, (256, 256)), (11008, 4096, 1025, (256, 256)), (2048, 8192, 8000, (256, 256)),
    (5760, 2944, 2560, (256, 256)), (5760, 2944, 1300, (256, 160)), (11008, 4096, 2048, (256, 192)),
])
def test_prefill_takes_the_tile_with_the_fewest_rounds(n: int, k: int, m: int, tile: tuple[int, int]) -> None:
    cfg = untuned_config(m, n, k, 128)
    assert (cfg.block_m, cfg.block_n, cfg.split_k) == (*tile, 1)
    assert cfg.num_stages == (3 if tile == (256, 256) else 8)
