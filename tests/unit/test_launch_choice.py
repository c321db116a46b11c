"""The operators' launch choice (resolver and Python body) on the CPU, for an MI355X that is not there:
what each call would launch and what its dispatch counter says."""

from __future__ import annotations

import pytest
import torch

from tokenforge.kernels import _lib, autotune, ops
from tokenforge.kernels.config import SPAN_32BIT, default_config, fill_split, ksplit_config, ksplit_rows
from tokenforge.kernels.metrics import KERNEL_CALLS

FAMILY_OF = {_lib.KERNEL_IDS[k]: ("hip_gemm" if k in ("gemm_mfma", "gemm_fp8") else "hip_gemv") for k in _lib.KERNEL_IDS}
DEV = torch.device("cuda", 0)


@pytest.fixture(autouse=True)
def _mi355x(monkeypatch: pytest.MonkeyPatch) -> None:
    monkeypatch.setattr(ops, "device_arch", lambda device: "gfx950")
    monkeypatch.setattr(ops, "_gpu_id", lambda device: "amd-gfx950-256cu")
    KERNEL_CALLS.reset()


@pytest.mark.parametrize("kind", [ops.KIND_LINEAR, ops.KIND_W4A8, ops.KIND_NORM_LINEAR])
@pytest.mark.parametrize(("n", "k", "g"), [(896, 896, 64), (3584, 3584, 128), (37888, 3584, 128), (1152, 4096, 32)])
def test_the_counter_names_the_family_that_runs(kind: int, n: int, k: int, g: int) -> None:
    for m in (1, 3, 5, 8, 9, 16, 17, 100, 300):
        fields = ops._resolve_launch(kind, _lib.EPILOGUE_NONE, m, n, k, g, 0)
        assert ops._FAMILIES[fields[7]] == FAMILY_OF[fields[0]], f"m={m}"
        if kind == ops.KIND_NORM_LINEAR:
            continue
        before = {lab: KERNEL_CALLS.value(kernel=lab, bucket=ops._BUCKET_LABELS[fields[8]]) for lab in ops._FAMILIES}
        cfg = ops._decide(DEV, m, n, k, g, w4a8=kind == ops.KIND_W4A8)
        after = {lab: KERNEL_CALLS.value(kernel=lab, bucket=ops._BUCKET_LABELS[fields[8]]) for lab in ops._FAMILIES}
        assert {lab: after[lab] - before[lab] for lab in after} == {
            lab: int(lab == ops._family(cfg)) for lab in after}, f"m={m}"


@pytest.mark.parametrize(("n", "k", "one_launch"), [
    (3584, 3584, True), (896, 896, True), (9728, 896, True), (4096, 4096, True), (4112, 3584, False),
    (9728, 1536, False), (3584, 4224, False), (37888, 3584, False)])
def test_w4a8_up_to_16_rows_decodes_while_staging_where_that_is_faster(n: int, k: int, one_launch: bool) -> None:
    for m in (9, 12, 16):
        cfg = ops._decide(DEV, m, n, k, 128, w4a8=True)
        assert (cfg.family == "gemv") == one_launch, f"m={m}: {cfg}"
        if one_launch:
            assert ops._resolve_launch(ops.KIND_W4A8, _lib.EPILOGUE_NONE, m, n, k, 128, 0)[9] == 0  # no workspace
    assert ops._decide(DEV, 17, n, k, 128, w4a8=True).ksplit


@pytest.mark.parametrize(("n", "k", "g"), [(1000, 1024, 32), (4096, 4096, 128), (5760, 2944, 32), (3584, 18944, 128)])
def test_no_k_split_once_the_row_tiles_fill_the_cus(n: int, k: int, g: int) -> None:
    for m in (4097, 9000, 20000, 70000):
        cfg = ops._gpu_config(DEV, m, n, k, g)
        tiles = -(-m // cfg.block_m) * -(-n // cfg.block_n)
        assert cfg.split_k == 1 or tiles < 256, f"m={m}: {cfg}"
        need = ops._resolve_launch(ops.KIND_LINEAR, _lib.EPILOGUE_NONE, m, n, k, g, 0)[9]
        assert (need == 0) == (cfg.split_k == 1), f"m={m}"


def test_an_entry_of_the_callers_own_cache_keeps_its_tile() -> None:
    n, k, g = 37888, 3584, 128
    shipped = ops._gpu_config(DEV, 80, n, k, g)
    own = ksplit_config(4, 5, 4)
    autotune.get_cache("amd-gfx950-256cu").put(128, n, k, g, own)
    assert ops._gpu_config(DEV, 80, n, k, g) == ksplit_rows(own, 80) != shipped


def test_down_proj_at_256_rows_fills_the_cus_once() -> None:
    cfg = ops._gpu_config(DEV, 256, 3584, 18944, 128)
    assert (cfg.block_m, cfg.block_n, cfg.num_stages) == (256, 128, 8)
    assert cfg.split_k == fill_split(cfg, 256, 3584, 18944) == 9


def test_gate_up_keeps_its_columns_up_to_64_rows() -> None:
    for m in (9, 16, 17, 32, 33, 48, 49, 56, 63, 64):
        cfg = ops._gpu_config(DEV, m, 37888, 3584, 128)
        assert (cfg.block_n, cfg.waves_k, cfg.split_k) == (160, 4, 1), f"m={m}"
        assert cfg.block_m == 16 * -(-m // 16), f"m={m}"


def test_rows_past_32_bit_offsets_leave_a_tuned_tile() -> None:
    n, k, g = 1024, 1024, 32
    autotune.get_cache("amd-gfx950-256cu").put(256, n, k, g, ksplit_config(3, 4, 4))
    assert ops._gpu_config(DEV, 200, n, k, g, SPAN_32BIT - 2).ksplit
    assert ops._gpu_config(DEV, 200, n, k, g, SPAN_32BIT) == default_config(256, n, k, g)
