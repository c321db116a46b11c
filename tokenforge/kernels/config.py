"""M buckets and launch configurations of the gfx950 W4A16 kernels.

Counterpart of the reference's ``config.py`` (config.py:8-117). Differences, each forced by
the hardware or by the single HIP path:

* ``M_BUCKETS`` runs up to 4096: every M, prefill included, is served by a HIP kernel chosen
  through the bucket's autotune entry (the reference sends M > 128 to dequant + cuBLAS).
* ``GemmConfig`` names a compiled kernel variant: ``kernel`` is one of ``KERNELS`` and the
  tuple ``(kernel, block_m, block_n, block_k, num_warps, num_stages)`` must be in
  ``VARIANTS`` (the table ``libtokenforge_hip.so`` exports; a CPU test keeps the two equal).
  ``split_k`` is a runtime value.

Field meaning per kernel family:

========== =========================== ================================================
kernel     block_m / block_n / block_k  split_k / num_warps / num_stages
========== =========================== ================================================
gemv_dot   max M (1,2,4) / columns per  1 / waves per workgroup / 128-wide K steps in
           workgroup (16*RT) / 128 or   flight per wave; block_k as for gemv_mfma
           256
gemv_mfma  M per tile (16,32) / columns 1 / waves per workgroup / 128-wide K steps in
           per workgroup (16*RT) / 128  flight per wave. block_k 128: the waves split
           or 256                       K over the same columns and add their partials
                                        on chip; block_k 256: the waves take different
                                        column sets (block_n each) over the whole K and
                                        share one staged x
gemv_mfma  max M (4) / 16 / 512: the    1 / waves per workgroup / steps in flight per wave.
(stream)   stream form                  Workgroups own tile ranges sized so the grid is
                                        resident; their waves take the range's 128-wide
                                        steps round robin (neighbouring blocks in flight)
gemm_mfma  LDS tile M / tile N / tile K K slices across workgroups (fp32 workspace,
                                        fixed-order reduce) / 4, 8 or 16 waves / 2: two
                                        LDS buffers, 3 and 4: pipelined with 2 and 3 x
                                        stages, 6 and 7: the same on 16x16 MFMA fragments
                                        (block_k 64); block_k 128: skinny form, num_stages
                                        = x stages (wave-tile form: 4 + x stages)
gemm_mfma  tile M (16..128) / tile N /  K slices across workgroups / 8 / 6, 7, 8: 2, 4, 8 of the
(K split)  128                          waves along K, the rest along N; weights go from memory to the
                                        MFMA, x through LDS
gemm_fp8   LDS tile M / tile N / 128    as gemm_mfma (8 waves, num_stages = x stages +
           (one group per block)        1). W4A8 only: e4m3 x on the fp8 MFMA, the group
                                        scale applied in fp32 after each group; chosen by
                                        ``fp8_gemm_config``, not by the W4A16 tuner
========== =========================== ================================================

Every kernel reads the weights in the gfx950 tile layout that ``pack.pack_awq`` produces.
"""

from __future__ import annotations

import functools
import math
from dataclasses import asdict, dataclass, replace
from typing import Any

M_BUCKETS: tuple[int, ...] = (1, 2, 4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048, 4096)
MAX_BUCKET_M = M_BUCKETS[-1]
GEMV_MAX_M = 32
"""Largest bucket the streaming (gemv) kernels serve; by default larger ones use the GEMM."""
GEMM_MIN_M = 16
"""Smallest bucket the gemm_mfma kernels may serve (the tuner weighs both families at 16, 32)."""

KERNELS: tuple[str, ...] = ("gemv_dot", "gemv_mfma", "gemm_mfma", "gemm_fp8")
NUM_CUS = 256
"""MI355X compute units; the split heuristics aim to put several waves on each."""

_WAVES = (1, 2, 4, 8, 16)

# Compiled streaming variants: (kernel, block_m, column tiles RT, block_k, ring depth P, max
# waves). block_k = 128: the waves of a workgroup split K and x is staged in LDS per wave;
# block_k = 256: the waves take different column tiles over the whole K and share one copy of
# x. The wave cap keeps each variant within the VGPR budget of its launch bound (no spills).
GEMV_TEMPLATES: tuple[tuple[str, int, int, int, int, int], ...] = (
    ("gemv_dot", 1, 1, 128, 2, 16), ("gemv_dot", 1, 1, 128, 4, 16), ("gemv_dot", 1, 2, 128, 2, 16),
    ("gemv_dot", 2, 1, 128, 2, 16), ("gemv_dot", 4, 1, 128, 2, 16),
    ("gemv_dot", 1, 1, 256, 2, 8), ("gemv_dot", 1, 1, 256, 4, 8), ("gemv_dot", 2, 1, 256, 4, 8),
    ("gemv_dot", 4, 1, 256, 4, 8),
    ("gemv_mfma", 16, 1, 128, 2, 16), ("gemv_mfma", 16, 1, 128, 4, 16), ("gemv_mfma", 16, 1, 128, 8, 16),
    ("gemv_mfma", 16, 2, 128, 2, 16), ("gemv_mfma", 16, 2, 128, 4, 8), ("gemv_mfma", 16, 4, 128, 2, 8),
    ("gemv_mfma", 32, 1, 128, 2, 16), ("gemv_mfma", 32, 2, 128, 2, 8),
    ("gemv_mfma", 16, 1, 256, 2, 8), ("gemv_mfma", 16, 1, 256, 4, 8), ("gemv_mfma", 16, 1, 256, 8, 8),
    ("gemv_mfma", 16, 2, 256, 2, 8), ("gemv_mfma", 16, 2, 256, 4, 8), ("gemv_mfma", 32, 1, 256, 2, 8),
)


def _gemv_variants() -> list[tuple[str, int, int, int, int, int]]:
    out = []
    for kernel, bm, rt, bk, stages, max_waves in GEMV_TEMPLATES:
        out += [(kernel, bm, 16 * rt, bk, w, stages) for w in _WAVES if w <= max_waves]
    return out


STREAM_BLOCK_K = 512
"""``block_k`` of the GEMV stream form (gemv_mfma, M <= its block_m)."""
STREAM_MAX_M = 4
"""block_m of the stream form that serves M <= 4 (and runs the RMSNorm prologue)."""
STREAM_WIDE_M = 8
"""block_m of the stream form that serves the bucket of M = 5..8 (no RMSNorm prologue)."""
STREAM_MAX_X_BYTES = 96 * 1024
"""The stream form stages x in LDS: M rows of K + 8 fp16 values (of K / split_k + 8 under a K
split) must fit this."""
STREAM_SPLITS = (2, 4)
"""K splits the tuner tries on the stream form (split_k 1 besides): each workgroup stages and
multiplies one K slice, the split-K reduce adds the slices."""


def _stream_variants() -> list[tuple[str, int, int, int, int, int]]:
    # block_m 4: ring depth 2 and 4, every wave count; block_m 8: 4, 8 or 16 waves.
    return ([("gemv_mfma", STREAM_MAX_M, 16, STREAM_BLOCK_K, w, p) for p in (2, 4) for w in _WAVES]
            + [("gemv_mfma", STREAM_WIDE_M, 16, STREAM_BLOCK_K, w, p) for p in (2, 4) for w in (4, 8, 16)])


NORM_MAX_K = 8192
"""Largest K whose RMSNorm the GEMV stream form runs in its prologue."""


def norm_scratch_bytes(m: int, k: int) -> int:
    """LDS the stream form's RMSNorm prologue adds: M rows of chunk sums (fp64), each padded to
    the power of two >= K / 8 (at least 64), 256 bytes of maxima and the staged norm weight
    (K fp16)."""
    lpad = 64
    while lpad < k // 8:
        lpad *= 2
    return m * lpad * 8 + 256 + 2 * k


def stream_slice_k(k: int, split_k: int) -> int:
    """K of the longest slice when the stream form splits K over ``split_k`` workgroup sets."""
    return -(-(k // 128) // split_k) * 128


def stream_form_applies(m: int, n: int, k: int, num_warps: int, norm: bool = False,
                        max_m: int = STREAM_MAX_M, split_k: int = 1) -> bool:
    """Whether the op runs a call of this shape on the GEMV stream form when its bucket's config
    is that form (``max_m``: the config's block_m, ``split_k``: its K split): M <= max_m, N % 32
    == 0, K % 128 == 0 with at least one 128-wide step per wave in every K slice, and the
    slice of x small enough to stage in LDS. The rule does not depend on the epilogue, so a
    plain call and its fused SiLU*mul or residual twin run the same kernel and agree bit for bit
    (the library itself runs plain and residual calls on N % 16 == 0 as well). With ``norm``
    (the RMSNorm prologue of ``rmsnorm_fp8_w4a16_linear``, on the block_m 4 form without a K
    split only) M is at most 4, K at most NORM_MAX_K and the staged x plus the prologue's
    scratch must fit."""
    if k % 128 or split_k < 1:
        return False
    x_bytes = m * (stream_slice_k(k, split_k) + 8) * 2 + (norm_scratch_bytes(m, k) if norm else 0)
    return (
        1 <= m <= (STREAM_MAX_M if norm else max_m)
        and n % 32 == 0
        and (k // 128) // split_k >= num_warps
        and x_bytes <= STREAM_MAX_X_BYTES
        and (not norm or (k <= NORM_MAX_K and split_k == 1))
    )


NORM_FUSED_MAX_M = 1
"""``rmsnorm_fp8_w4a16_linear`` runs the norm inside the GEMV (its prologue) up to this M. Measured
on MI355X (qkv and gate_up of Qwen2.5-7B): at M = 1 the prologue saves the norm kernel's launch
(qkv 9.7 us against 7.3 + 3.5 for the two kernels); at M = 2 and 4 every workgroup's norm of
several rows takes longer than the separate norm kernel (qkv M = 4: 16.2 us against 11.6)."""
NORM_RING_DEPTH = 4
"""Ring depth (num_stages) of the stream form when it runs the RMSNorm prologue: the loads in
flight while the prologue runs keep HBM busy (qkv M = 1: 9.7 us at depth 4 against 10.5 at 2;
gate_up 19.9 against 21.3; depth 8 no better)."""


def norm_fused_config(cfg: GemmConfig, m: int, n: int, k: int) -> GemmConfig | None:
    """The config ``rmsnorm_fp8_w4a16_linear`` runs the fused kernel on, given the bucket's
    ``cfg``, or None where it runs the norm kernel and the linear: M <= NORM_FUSED_MAX_M, a
    stream-form config of block_m 4 without a K split, and the prologue fits
    (``stream_form_applies(norm=True)``); the ring deepened to NORM_RING_DEPTH. Both routes give
    the same bits."""
    if not (1 <= m <= NORM_FUSED_MAX_M and cfg.stream and cfg.block_m == STREAM_MAX_M and cfg.split_k == 1):
        return None
    if not stream_form_applies(m, n, k, cfg.num_warps, norm=True):
        return None
    return replace(cfg, num_stages=max(cfg.num_stages, NORM_RING_DEPTH))


def _gemm_variants() -> list[tuple[str, int, int, int, int, int]]:
    # num_stages 2: two LDS buffers, operands staged through registers (any group size).
    tiles = [(64, 64, 64), (64, 128, 64), (128, 64, 64), (128, 128, 64), (128, 256, 64),
             (256, 128, 64), (256, 256, 64), (64, 64, 32), (128, 128, 32), (256, 128, 32)]
    out = [("gemm_mfma", bm, bn, bk, 4, 2) for bm, bn, bk in tiles]
    # num_stages 3 / 4: pipelined form, x streamed into 2 / 3 LDS stages, weights prefetched two
    # blocks ahead (block_k 64, group size 64 or 128); 4 or 8 waves.
    tiles3 = [(256, 160), (256, 128), (128, 256), (128, 128), (256, 192), (256, 96), (64, 256), (128, 192)]
    out += [("gemm_mfma", bm, bn, 64, 4, 4) for bm, bn in tiles3]
    out += [("gemm_mfma", 256, 256, 64, 8, 3), ("gemm_mfma", 256, 192, 64, 8, 3),
            ("gemm_mfma", 256, 192, 64, 8, 4), ("gemm_mfma", 256, 128, 64, 8, 3),
            ("gemm_mfma", 128, 256, 64, 8, 3), ("gemm_mfma", 256, 160, 64, 8, 3)]
    # ... and 16 waves (four per SIMD), 32-row wave tiles.
    out += [("gemm_mfma", 256, 192, 64, 16, 3), ("gemm_mfma", 256, 192, 64, 16, 4), ("gemm_mfma", 256, 128, 64, 16, 3)]
    # num_stages 6 / 7: the same pipeline on 16x16 MFMA fragments (16-column wave-tile
    # granularity): 256 x 160 tiles with 16 or 8 waves, 256 x 128 .. 256 with 8, 128-row tiles
    # with 4 or 8.
    out += [("gemm_mfma", 256, 160, 64, 16, 6), ("gemm_mfma", 256, 160, 64, 16, 7), ("gemm_mfma", 256, 160, 64, 8, 6),
            ("gemm_mfma", 256, 160, 64, 8, 7), ("gemm_mfma", 256, 192, 64, 8, 6), ("gemm_mfma", 256, 224, 64, 8, 6),
            ("gemm_mfma", 256, 128, 64, 8, 6), ("gemm_mfma", 256, 256, 64, 8, 6), ("gemm_mfma", 128, 160, 64, 4, 6),
            ("gemm_mfma", 128, 128, 64, 4, 6), ("gemm_mfma", 128, 256, 64, 8, 6)]
    # num_stages 8: the producer / consumer form (two x stages): num_warps consumer waves only
    # read fragments and run MFMAs, four producer waves stage x and dequantize the weights.
    out += [("gemm_mfma", 256, 160, 64, 8, 8), ("gemm_mfma", 256, 128, 64, 8, 8), ("gemm_mfma", 128, 256, 64, 8, 8),
            ("gemm_mfma", 128, 128, 64, 4, 8), ("gemm_mfma", 256, 192, 64, 8, 8)]
    # block_k 128: skinny form (M <= 128), weights streamed into MFMA registers, 4 waves,
    # num_stages = x stages in LDS.
    skinny = [(1, 1, 3), (1, 2, 3), (1, 4, 3), (2, 1, 3), (2, 2, 3), (2, 4, 3), (4, 1, 3), (4, 2, 3),
              (4, 4, 3), (8, 1, 3), (8, 2, 3), (2, 2, 2), (4, 2, 2)]
    out += [("gemm_mfma", 16 * mt, 64 * rt, 128, 4, st) for mt, rt, st in skinny]
    # ... and with two waves along M: 256 x 160 tiles (gate_up at M >= 256: 237 tiles).
    out += [("gemm_mfma", 256, 160, 128, 4, 2)]
    # block_k 128, num_stages 4 + S: the wave-tile form (one wave per SIMD, 16 MT x 16 RT per
    # wave, WM waves along M), S x stages (x issued S - 1 steps ahead, weights three).
    wave_tiles = [(8, 5, 1, 3), (8, 4, 1, 4), (8, 3, 1, 4), (8, 2, 1, 4)]
    out += [("gemm_mfma", 16 * mt * wm, 16 * rt * (4 // wm), 128, 4, 4 + st) for mt, rt, wm, st in wave_tiles]
    # block_k 128, eight waves: the K-split tile form, 8 / WK waves along N and WK along K, 16 MT rows
    # x 16 RT (8 / WK) columns; num_stages 6, 7, 8 for WK = 2, 4, 8.
    out += [ksplit_config(mt, rt, wk).variant() for mt, rt, wk in KSPLIT_TILES]
    return out


KSPLIT_TILES: tuple[tuple[int, int, int], ...] = (
    (1, 1, 8), (1, 2, 8), (1, 4, 8), (2, 1, 8), (2, 2, 8), (2, 4, 8),
    (1, 2, 4), (1, 4, 4), (1, 5, 4), (2, 2, 4), (2, 4, 4), (2, 5, 4), (3, 2, 4), (3, 4, 4), (3, 5, 4), (4, 2, 4),
    (4, 4, 4), (4, 5, 4), (2, 2, 2), (3, 3, 2), (4, 2, 2), (4, 3, 2), (5, 3, 2), (6, 2, 2), (6, 3, 2), (8, 1, 2), (8, 2, 2),
)
"""The K-split tile form's (row fragments MT, column tiles per wave RT, waves along K WK), in the
library's order."""


def ksplit_config(mt: int, rt: int, wk: int, split_k: int = 1) -> GemmConfig:
    """The K-split tile config of 16 ``mt`` rows x 16 ``rt`` (8 / ``wk``) columns."""
    return GemmConfig("gemm_mfma", 16 * mt, 16 * rt * (8 // wk), 128, split_k, 8, {2: 6, 4: 7, 8: 8}[wk])


# W4A8 fp8 GEMM tiles (block_m, block_n, waves along M, waves along N, x stages), in the
# library's order.
FP8_TILES: tuple[tuple[int, int, int, int, int], ...] = (
    (256, 192, 4, 2, 2), (256, 128, 4, 2, 2), (128, 256, 2, 4, 2), (256, 160, 4, 2, 2), (128, 128, 2, 4, 2),
    (256, 192, 4, 2, 3),
)


FP8_PC_TILES: tuple[tuple[int, int, int, int], ...] = ((256, 160, 4, 2), (256, 128, 4, 2), (128, 256, 2, 4), (128, 128, 2, 4))
"""The fp8 GEMM's producer / consumer form (num_stages 8): (block_m, block_n, consumer waves
along M, along N), in the library's order after FP8_TILES."""


def _fp8_variants() -> list[tuple[str, int, int, int, int, int]]:
    return ([("gemm_fp8", bm, bn, 128, wm * wn, s + 1) for bm, bn, wm, wn, s in FP8_TILES]
            + [("gemm_fp8", bm, bn, 128, wm * wn, 8) for bm, bn, wm, wn in FP8_PC_TILES])


def m_bucket(m: int) -> int:
    """Smallest bucket >= m (config.py:13-20). M above the largest bucket uses the largest."""
    if m < 1:
        raise ValueError(f"M must be >= 1, got {m}")
    for b in M_BUCKETS:
        if m <= b:
            return b
    raise ValueError(f"M={m} exceeds the largest bucket ({MAX_BUCKET_M})")


def family_for_bucket(bucket: int) -> str:
    """Default family of a bucket: ``gemv`` below GEMM_MIN_M, ``gemm`` from it on (the tuner
    may still pick a gemv kernel up to GEMV_MAX_M)."""
    return "gemv" if bucket < GEMM_MIN_M else "gemm"


@dataclass(frozen=True)
class GemmConfig:
    kernel: str
    block_m: int
    block_n: int
    block_k: int
    split_k: int = 1
    num_warps: int = 4
    num_stages: int = 2

    @property
    def path(self) -> str:
        return self.kernel

    @property
    def skinny(self) -> bool:
        """The register-streamed gemm_mfma forms (block_k 128), which read each lane's group
        themselves."""
        return self.kernel == "gemm_mfma" and self.block_k == 128

    @property
    def ksplit(self) -> bool:
        """The K-split tile form of gemm_mfma (block_k 128, eight waves)."""
        return self.skinny and self.num_warps == 8

    @property
    def waves_k(self) -> int:
        """Waves along K of the K-split tile form: num_stages 6, 7, 8 for 2, 4, 8."""
        return 1 << (self.num_stages - 5)

    @property
    def stream(self) -> bool:
        """The GEMV stream form (gemv_mfma, block_k 512), which serves M <= 4."""
        return self.kernel == "gemv_mfma" and self.block_k == STREAM_BLOCK_K

    @property
    def family(self) -> str:
        return "gemm" if self.kernel in ("gemm_mfma", "gemm_fp8") else "gemv"

    def variant(self) -> tuple[str, int, int, int, int, int]:
        return (self.kernel, self.block_m, self.block_n, self.block_k, self.num_warps, self.num_stages)

    def validate(self, group_size: int) -> None:
        """Raise ``ValueError`` if this config cannot run for ``group_size``."""
        if self.kernel not in KERNELS:
            raise ValueError(f"kernel={self.kernel!r} not in {KERNELS}")
        if self.kernel == "gemm_mfma" and not self.skinny and (
            self.block_k <= 0 or self.block_k > group_size or group_size % self.block_k
        ):
            raise ValueError(f"block_k={self.block_k} must divide group_size={group_size}")
        if not 1 <= self.split_k <= 16:
            raise ValueError(f"split_k={self.split_k} must be in [1, 16]")
        if self.family != "gemm" and not self.stream and self.split_k != 1:
            raise ValueError(
                f"split_k={self.split_k}: {self.kernel} splits K across its num_warps waves; "
                "split_k must be 1"
            )
        if self.num_warps not in _WAVES:
            raise ValueError(f"num_warps={self.num_warps} must be a power of two <= 16")
        if not 1 <= self.num_stages <= 8:
            raise ValueError(f"num_stages={self.num_stages} must be in [1, 8]")
        if self.variant() not in _VARIANT_SET:
            raise ValueError(f"{self.variant()} is not a compiled variant (block_m/block_n/block_k)")

    def fits_bucket(self, bucket: int) -> bool:
        """Whether this config may serve M values of ``bucket`` (cache validation): the gemv
        kernels serve buckets up to GEMV_MAX_M (gemv_dot and the stream form only up to their
        block_m), gemm_mfma buckets from GEMM_MIN_M on."""
        if self.family == "gemm":
            return bucket >= GEMM_MIN_M
        if bucket > GEMV_MAX_M:
            return False
        if self.stream:  # block_m 4 serves buckets up to 4, block_m 8 the bucket above
            return bucket <= self.block_m and (self.block_m == STREAM_MAX_M or bucket > STREAM_MAX_M)
        return self.kernel != "gemv_dot" or self.block_m >= bucket

    def to_dict(self) -> dict[str, Any]:
        return asdict(self)

    @classmethod
    def from_dict(cls, d: Any) -> GemmConfig:
        if not isinstance(d, dict):
            raise TypeError(f"config must be an object, got {type(d).__name__}")
        fields = set(cls.__dataclass_fields__)
        unknown = set(d) - fields
        if unknown:
            raise ValueError(f"unknown config keys {sorted(unknown)}")
        if not isinstance(d.get("kernel"), str):
            raise TypeError("config 'kernel' must be a string")
        ints = {k: v for k, v in d.items() if k != "kernel"}
        if not all(isinstance(v, int) and not isinstance(v, bool) for v in ints.values()):
            raise TypeError("config values must be integers")
        return cls(**d)


VARIANTS: tuple[tuple[str, int, int, int, int, int], ...] = tuple(
    _gemv_variants() + _stream_variants() + _gemm_variants() + _fp8_variants()
)
"""(kernel, block_m, block_n, block_k, num_warps, num_stages), in the library's order."""
_VARIANT_SET = frozenset(VARIANTS)


def _pow2_at_most(v: int, cap: int) -> int:
    p = 1
    while p * 2 <= min(v, cap):
        p *= 2
    return p


def split_k_gemv_config(n: int, k: int) -> GemmConfig:
    """The GEMV form that runs every shape (K split over the waves of a workgroup): one
    workgroup per 32 output columns, waves added until the grid holds about 12 per CU, never
    more waves than 128-wide K steps."""
    tiles = -(-n // 32)
    k_steps = max(1, -(-k // 128))
    waves = _pow2_at_most(max(1, -(-(12 * NUM_CUS) // tiles)), min(16, k_steps))
    return GemmConfig("gemv_mfma", 16, 32, 128, 1, waves, 2)


def default_config(bucket: int, n: int, k: int, group_size: int) -> GemmConfig:
    """Heuristic config used before tuning (config.py:71-92, re-derived for 256 CUs).

    Streaming kernels (M < 16): for M <= 4 the stream form with 8 waves and a ring of 2 where
    it applies; otherwise one workgroup per 32 output columns, adding
    waves (on-chip K slices) until the grid holds about 12 waves per CU, never more waves than
    128-wide K steps.
    Skinny GEMM (16 <= M <= 128): 16-64 rows x 64 or 128 columns per workgroup, K split until
    the grid holds about 1.5 workgroups per CU.
    Pipelined GEMM (M >= 256, group >= 64): 256 x 192 tiles of 8 waves (256 x 256 from M 1024);
    two-buffer GEMM for group 32.
    """
    if family_for_bucket(bucket) == "gemv":
        if bucket <= STREAM_MAX_M and stream_form_applies(bucket, n, k, 8):
            return GemmConfig("gemv_mfma", STREAM_MAX_M, 16, STREAM_BLOCK_K, 1, 8, 2)
        return split_k_gemv_config(n, k)
    if bucket <= 128:
        bm = min(bucket, 64)
        bn = 64 if bucket <= 64 else 128
        tiles = -(-n // bn) * -(-bucket // bm)
        k_steps = max(1, -(-k // 128))
        split = 1
        while tiles * split * 2 <= 3 * NUM_CUS and split * 2 <= min(8, k_steps):
            split *= 2
        return GemmConfig("gemm_mfma", bm, bn, 128, split, 4, 3)
    if group_size >= 64:
        bm, bn = (256, 192) if bucket <= 512 else (256, 256)
        tiles = -(-n // bn) * -(-bucket // bm)
        k_blocks = k // 64
        split = 1
        while tiles * split < NUM_CUS and split * 2 <= min(8, k_blocks):
            split *= 2
        return GemmConfig("gemm_mfma", bm, bn, 64, split, 8, 3)
    block_k = 64 if group_size >= 64 else 32
    if bucket <= 64:
        bm, bn = 64, 64
    elif bucket <= 128:
        bm, bn = 128, 128
    else:
        bm, bn = (256, 128) if block_k == 64 else (256, 128)
    tiles = -(-n // bn) * -(-bucket // bm)
    k_blocks = k // block_k
    split = 1
    while tiles * split < NUM_CUS and split * 2 <= min(16, k_blocks):
        split *= 2
    return GemmConfig("gemm_mfma", bm, bn, block_k, split, 4, 2)


# ----------------------------------------------------------------------------- untuned launches

SPAN_32BIT = 1 << 31
"""Bytes of x and of the packed weights from which on only the two-buffer GEMM (num_stages 2) runs: the
other kernels address both through 32-bit buffer offsets."""


def ksplit_applies(n: int, k: int) -> bool:
    """Whether a layer can run on the K-split tile form: whole 16-column tiles and 128-wide K steps."""
    return n % 16 == 0 and k % 128 == 0


def ksplit_rows(cfg: GemmConfig, m: int) -> GemmConfig:
    """A K-split tile config with the fewest compiled rows that cover M in as many tiles, its
    columns and waves along K unchanged (so every sum keeps its order): a bucket's config is tuned
    at the bucket's M, and rows past M cost LDS reads and MFMAs like any other (gate_up at M = 48 in
    the bucket of 64: 23.5 us with 48 rows, 25.9 with 64)."""
    tiles = -(-m // cfg.block_m)
    rows = [v[1] for v in VARIANTS
            if v[0] == cfg.kernel and v[2:] == cfg.variant()[2:] and v[1] <= cfg.block_m and -(-m // v[1]) == tiles]
    return replace(cfg, block_m=min(rows)) if rows else cfg


# Time model of the GEMM forms an untuned layer can run on, in microseconds and bytes:
#   T = launch + (work^q + hbm^q + l2^q)^(1/q) [+ split], work = rounds over the CUs x time of one
# workgroup; hbm the layer, x and y once; l2 every workgroup's weights and x. A K-split workgroup runs
# iterations of MFMAs (MT RT), dequantization (RT) and x (MT WK); an LDS-tile one K blocks of 64 and a
# skinny one K steps of 128 at its tile's rate. Fitted (least squares over log time) to launches of every
# tile and split on ten layer shapes from 1152 x 896 to 37888 x 3584, M = 16 .. 2048, on MI355X; the two
# tiles that were the defaults before were added beside it. bench_probes/launch_choice.py checks the
# choice against those defaults and gives the data of a refit. Over 11295 calls on 1465 random layers (M
# = 1 .. 8000, cold weights) it takes 0.45 to 0.88 of the default's time in the mean of a range of M; 69
# calls are more than 3% slower, at most 1.25 times. The modelled time is 0.84 (M > 4096) to 1.0 of the measured
# one, with a spread of 9 to 16%.
_NUM = {
    "launch": 1.73, "q": 1.66, "hbm": 7.57e6, "split": 2.26, "partials": 8.74e6,
    "ks_wg": 2.49, "mfma": 0.0836, "dequant": 0.172, "x": 0.0065, "pair": 1.27, "ks_l2": 25.6e6,
    "pc_wg": 5.53, "pc_block": 0.130, "pc_l2": 17.0e6,
    # one 64-K block of a tile
    "pc": {(256, 192): 0.917, (256, 160): 0.803, (256, 128): 0.512, (128, 256): 0.658, (128, 128): 0.192},
    # the shared-role 256 x 256 tile, fitted to 880 launches above M = 256 beside the others' model
    "wide_wg": 7.0, "wide_block": 1.52,
    # the default of 9 .. 32 rows (16 or 32 x 64, no LDS sums), fitted to 1640 launches the same way
    "skinny_wg": 2.0, "skinny_step": 0.35, "skinny_l2": 50e6,
}


@dataclass(frozen=True)
class _Cost:
    """A tile's constants in the time model."""

    wg_us: float  # prologue and end of a workgroup
    iter_us: float  # an iteration (K split), a block of 64 or a step of 128 K
    l2_rate: float  # bytes of its loads per us
    per_cu: int = 1  # workgroups a CU holds ...
    share: float = 1.0  # ... and the time of a round of them beside one workgroup's


@functools.lru_cache(maxsize=None)
def _model_tiles(group_size: int, ksplit: bool) -> tuple[tuple[GemmConfig, _Cost], ...]:
    """The model's candidate tiles (split_k 1) and their constants."""
    out = []
    for mt, rt, wk in KSPLIT_TILES if ksplit else ():
        per_iter = _NUM["mfma"] * mt * rt + _NUM["dequant"] * rt + _NUM["x"] * mt * wk
        pair = mt * rt <= 4 and rt <= 2 and mt * wk <= 8  # registers and LDS of a second workgroup
        cost = _Cost(_NUM["ks_wg"], per_iter, _NUM["ks_l2"], 2 if pair else 1, _NUM["pair"] if pair else 1.0)
        out.append((ksplit_config(mt, rt, wk), cost))
    if group_size >= 64:
        for (bm, bn), tile in _NUM["pc"].items():
            w = 4 if (bm, bn) == (128, 128) else 8
            out.append((GemmConfig("gemm_mfma", bm, bn, 64, 1, w, 8),
                        _Cost(_NUM["pc_wg"], _NUM["pc_block"] + tile, _NUM["pc_l2"])))
        # Slower per column than the producer/consumer tiles but wider than any of them: the fewest
        # rounds where its tiles fill one or two (4096 x 4096 M = 3584 124 us, 256 x 128 133).
        out.append((GemmConfig("gemm_mfma", 256, 256, 64, 1, 8, 3),
                    _Cost(_NUM["wide_wg"], _NUM["wide_block"], _NUM["pc_l2"])))
    return tuple(out)


def _model_us(cfg: GemmConfig, cost: _Cost, m: int, n: int, k: int) -> float:
    """Modelled time of ``cfg`` (a tile with a split)."""
    q, split = _NUM["q"], cfg.split_k
    wgs = -(-m // cfg.block_m) * -(-n // cfg.block_n) * split
    if wgs <= NUM_CUS:
        rounds = 1.0
    else:
        rounds = -(-wgs // (cost.per_cu * NUM_CUS)) * cost.share
    steps = -(-(k // 128) // split)
    iters = -(-steps // cfg.waves_k) if cfg.ksplit else steps if cfg.skinny else 2 * steps
    work = rounds * (cost.wg_us + iters * cost.iter_us)
    l2 = wgs * (cfg.block_n * 0.53 + cfg.block_m * 2) * (k / split) / cost.l2_rate
    hbm = (n * k * 0.53 + m * k * 2 + m * n * 2) / _NUM["hbm"]
    us = _NUM["launch"] + (work**q + hbm**q + l2**q) ** (1 / q)
    return us + (_NUM["split"] + split * m * n * 8 / _NUM["partials"] if split > 1 else 0.0)


@functools.lru_cache(maxsize=4096)
def _modelled_config(m: int, n: int, k: int, group_size: int) -> tuple[float, GemmConfig] | None:
    """The modelled time and config of the fastest tile and split (None: no form serves the layer)."""
    best: tuple[float, GemmConfig] | None = None
    steps = k // 128
    for cfg, cost in _model_tiles(group_size, ksplit_applies(n, k)):
        if cfg.ksplit and (m <= cfg.block_m - 16 or (-(-m // cfg.block_m) > 4 if m <= 128 else
                                                     cfg.block_m < 48 or cfg.block_n < 64)):
            continue  # a smaller tile holds M, or outside the fit: many small tiles refetch the weights
        tiles = -(-m // cfg.block_m) * -(-n // cfg.block_n)
        for split in (1, 2, 3, 4, 6, 8):
            if split > 1 and (tiles * split > 2 * NUM_CUS or steps < split * (cfg.waves_k if cfg.ksplit else 2)):
                break
            split_cfg = replace(cfg, split_k=split)
            us = _model_us(split_cfg, cost, m, n, k)
            if best is None or us < best[0]:
                best = (us, split_cfg)
    return best


def _model_rows(m: int) -> int:
    """M rounded up for the model: one evaluation per step of M, not per M."""
    unit = 16 if m <= 128 else 64 if m <= 1024 else 256
    return -(-m // unit) * unit


RETUNE_MARGIN = 0.93
"""A shipped K-split tile gives way to the modelled best at this M where the model puts that below
this share of the tuned tile's time: well inside a bucket the tuned columns can be the wrong ones.
Measured on MI355X on 88 calls inside the buckets (cold weights): of the 30 that give way 26 are 2 to
27% faster (gate_up M = 80 46.6 -> 34.5 us, qkv M = 300 25.2 -> 19.6), the four at down M = 33 .. 48
within 1%. Where M rounds up to the bucket's own rows the tuner has measured the very tiles and its
choice stands."""


@functools.lru_cache(maxsize=4096)
def _retiled(cfg: GemmConfig, m: int, n: int, k: int, group_size: int) -> GemmConfig:
    best = _modelled_config(m, n, k, group_size)
    tiles = {c.variant(): cost for c, cost in _model_tiles(group_size, True)}
    if best is None or cfg.variant() not in tiles:
        return cfg
    tuned = _model_us(cfg, tiles[cfg.variant()], m, n, k)
    return best[1] if best[0] < RETUNE_MARGIN * tuned else cfg


def tuned_at(cfg: GemmConfig, m: int, n: int, k: int, group_size: int, own: bool = False) -> GemmConfig:
    """The config of a call with M rows whose bucket is tuned to ``cfg``: a K-split tile loses the
    rows M does not need and, unless the caller's own tuner chose it (``own``) or M rounds up to the
    bucket's rows, may give way to the modelled best."""
    if not cfg.ksplit:
        return cfg
    cfg = ksplit_rows(cfg, m)
    if own or m > MAX_BUCKET_M or not ksplit_applies(n, k) or _model_rows(m) == _model_rows(m_bucket(m)):
        return cfg
    return _retiled(cfg, _model_rows(m), n, k, group_size)


def _narrow_decode_config(m: int, n: int, k: int, base: GemmConfig) -> GemmConfig:
    """The M <= 4 choice between ``base``, the bucket's default (the stream form, or the 32-column GEMV
    where that does not run), and the GEMV with 16 columns a workgroup.

    Against the stream form, which stages every row of x whole: at M = 1 base; at M = 2 the GEMV up to K =
    4096, with 4 waves up to K = 2048 and 8 above, at M = 3 up to K = 2432 and at M = 4 up to K = 2048, with
    4 waves up to K = 1024 and 8 above; and with 16 waves for longer K (from K = 7168 at M = 3 and 4) while
    its workgroups are one round over the CUs (N <= 4096). GEMV / stream in us, cold weights; weights in the Infinity
    Cache: M = 2 4608 x 4096 7.0 / 7.3; 6.1 / 7.0, 2048 x 8192 7.0 / 7.7; 6.1 / 6.6, M = 3 2048 x 1024 4.0 /
    4.3; 3.6 / 4.1, 4608 x 2048 5.3 / 6.1; 5.0 / 5.8, 2048 x 8192 8.0 / 8.1; 6.7 / 7.1. On the other side M
    = 2 5120 x 5632 9.2 / 8.6; 7.4 / 7.9 (8 waves), M = 3 2048 x 5632 6.7 / 6.2; 6.2 / 5.9, 5120 x 11008 15.2
    / 13.7; 11.8 / 11.4, 4608 x 4096 8.1 / 7.4; 6.5 / 7.0 (a model of such layers does not fit the cache).
    Against the 32-column GEMV: while it is one round always, with 4, 8 or 16 waves by K (528 x 4096, M =
    3 5.3 / 7.0; 3584 x 18944 in groups of 32 14.4 / 20.6); past that 4 waves below K = 4096 and 64M
    weights and 8 up to K = 8192, or any K where the 32-column grid is past one round too (6160 x 8192
    11.6 / 12.3, 8208 x 11008 23.4 / 29.2; 4608 x 18944 24.5 / 20.9, 16400 x 4096 14.8 / 14.4, 20432 x 3840
    at M = 4 18.8 / 16.5)."""
    steps = k // 128
    one_round = n <= 16 * NUM_CUS
    if base.stream and m == 1:
        waves = 0
    elif base.stream and m == 2:
        waves = 4 if steps <= 16 else 8 if steps <= 32 else 16 if one_round else 0
    elif base.stream:
        waves = 4 if steps <= 8 else 8 if steps <= (19 if m == 3 else 16) else 16 if one_round and steps >= 56 else 0
    elif one_round:
        waves = 4 if steps < 32 else 8 if steps < 56 else 16
    elif steps < 32:
        waves = 4 if n * k <= 64 << 20 else 0
    else:
        waves = 8 if n < 640 * 16 and (steps <= 64 or n > 32 * NUM_CUS) else 0
    return GemmConfig("gemv_mfma", 16, 16, 128, 1, min(waves, _pow2_at_most(steps, 16)), 2) if waves else base


def untuned_config(m: int, n: int, k: int, group_size: int, x_bytes: int = 0) -> GemmConfig:
    """Config of a call with M rows on a layer nobody has tuned (no cache or shipped entry).
    ``x_bytes``: the bytes from x's first element to its last, for rows with a stride of their own.

    * A layer or an x too large for 32-bit offsets, and up to M = 128 a layer without whole tiles and
      K steps: :func:`default_config` of the bucket. Past 2 GiB the library runs only the two-buffer
      GEMM among these (M > 128 in groups of 32) and refuses the others, whose offsets are 32-bit.
    * M <= 8, at least 640 tiles of 16 columns (work for every CU): the stream form where it runs, with 16
      waves from K = 4096 on (11040 x 5504, M = 3 9.6 us against 10.8 with 8).
    * M <= 4 below that: :func:`_narrow_decode_config`.
    * M = 5 .. 8: a wide layer of few weights as at M <= 4 (K too short for the stream form: 17712 x 256
      4.4 us against 5.7 for the tile), the others the modelled tile (512 x 4096 5.6 us against 8.2).
    * M > 8: the modelled best of the K-split, the producer/consumer and the 256 x 256 tiles; up to M = 32
      the bucket's default where the model puts that first (its tiles come three or two to a CU: 31200 x
      1408 M = 17 10.7 us against 11.9, 6144 x 13696 M = 11 17.0 against 18.8).
    """
    bucket = MAX_BUCKET_M if m > MAX_BUCKET_M else m_bucket(m)
    base = default_config(bucket, n, k, group_size)
    steps = k // 128
    ksplit = ksplit_applies(n, k)
    if n * k // 2 >= SPAN_32BIT or max(m * k * 2, x_bytes) >= SPAN_32BIT or steps < 2 or (not ksplit and m <= 128):
        return base
    if 1 < m <= STREAM_WIDE_M and n >= 640 * 16 and n % 32 == 0:
        form = GemmConfig("gemv_mfma", STREAM_MAX_M if m <= STREAM_MAX_M else STREAM_WIDE_M, 16, STREAM_BLOCK_K, 1,
                          16 if steps >= 32 else 8, 2)
        if stream_form_applies(m, n, k, form.num_warps, max_m=form.block_m):
            return form
    if m <= STREAM_MAX_M or (m <= STREAM_WIDE_M and n >= 640 * 16 and n * k <= 12 << 20):
        return _narrow_decode_config(m, n, k, base)
    best = _modelled_config(_model_rows(m), n, k, group_size)
    if best is None:
        return base
    if STREAM_WIDE_M < m <= 32:
        skinny = _Cost(_NUM["skinny_wg"], _NUM["skinny_step"], _NUM["skinny_l2"], 3 if base.block_m == 16 else 2)
        if _model_us(base, skinny, m, n, k) < best[0]:
            return base
    return best[1]


def candidate_configs(bucket: int, group_size: int) -> list[GemmConfig]:
    """Autotune search space for one bucket: every compiled variant that fits the bucket (both
    families for buckets GEMM_MIN_M..GEMV_MAX_M)."""
    out: list[GemmConfig] = []
    for kernel, bm, bn, bk, warps, stages in VARIANTS:
        if kernel == "gemm_fp8":  # W4A8 only (fp8_gemm_config), never a W4A16 candidate
            continue
        cfg = GemmConfig(kernel, bm, bn, bk, 1, warps, stages)
        if not cfg.fits_bucket(bucket):
            continue
        if cfg.family == "gemv":
            if kernel == "gemv_mfma" and bm > 16 and bucket <= 16:
                continue
            out.append(cfg)
            if cfg.stream:  # K split across workgroups: x rows of a long K staged by slices
                out.extend(replace(cfg, split_k=s) for s in STREAM_SPLITS)
            continue
        if bk != 128 and (bk > group_size or group_size % bk):
            continue
        if bm > 2 * bucket:
            continue
        out.extend(GemmConfig(kernel, bm, bn, bk, s, warps, stages) for s in (1, 2, 4, 8))
    return out


def fill_split(cfg: GemmConfig, m: int, n: int, k: int, cus: int = 256) -> int:
    """The K split that finishes an LDS-tile GEMM launch in the fewest K blocks per CU when its
    workgroups run in whole rounds over ``cus`` CUs: argmin over s of ceil(tiles * s / cus) *
    ceil(blocks / s), the smallest such s. E.g. down_proj (3584 x 18944) at M = 256 in 256 x 128
    tiles: 28 tiles, 296 blocks of 64, split 9 (252 workgroups, 33 blocks each) against split
    8's 37 blocks. s stays within 16, the K blocks, and K / (8 M): the fp32 partials (s * M * N *
    4 bytes, written and read back) are then no larger than the packed weights (N * K / 2), the
    traffic the split is meant to spread. The tuner times the candidate like any other."""
    tiles = -(-m // cfg.block_m) * -(-n // cfg.block_n)
    blocks = k // cfg.block_k
    best, best_cost = 1, None
    for s in range(1, max(1, min(16, blocks, k // (8 * m))) + 1):
        cost = -(-tiles * s // cus) * -(-blocks // s)
        if best_cost is None or cost < best_cost:
            best, best_cost = s, cost
    return best


def fill_split_candidates(cands: list[GemmConfig], bucket: int, n: int, k: int, cus: int = 256) -> list[GemmConfig]:
    """For every LDS-tile GEMM tile among ``cands``, its :func:`fill_split` config when the
    candidates do not already hold it (they split K in powers of two)."""
    have = {(c.kernel, c.block_m, c.block_n, c.block_k, c.num_warps, c.num_stages, c.split_k) for c in cands}
    out: list[GemmConfig] = []
    for c in cands:
        if c.kernel != "gemm_mfma" or c.skinny or c.split_k != 1:
            continue
        s = fill_split(c, bucket, n, k, cus)
        key = (c.kernel, c.block_m, c.block_n, c.block_k, c.num_warps, c.num_stages, s)
        if key not in have:
            have.add(key)
            out.append(replace(c, split_k=s))
    return out


FP8_MIN_BUCKET = 128
"""W4A8 calls from this M bucket on run the fp8 GEMM (where it applies); smaller M stay on the
kernels that read the weights once per call (GEMV, skinny GEMM), which decode the codes to fp16."""


def fp8_gemm_applies(bucket: int, n: int, k: int, group_size: int) -> bool:
    """Whether a W4A8 call of this shape runs on the fp8 GEMM: prefill M, group_size 128,
    K % 128 == 0 and N % 16 == 0 (what ``gemm_fp8`` requires)."""
    return bucket >= FP8_MIN_BUCKET and group_size == 128 and k % 128 == 0 and n % 16 == 0


W4A8_GEMV_MAX_M = 16
"""Rows of one tile of the 16-column GEMV, up to which it may replace a K-split tile in a W4A8 call."""


def w4a8_gemv_config(m: int, n: int, k: int) -> GemmConfig | None:
    """The GEMV that a W4A8 call of M rows runs where its W4A16 config is a K-split tile, or None where
    the tile is the faster one. The GEMV decodes the codes while it stages x; the tile form has them
    converted to fp16 by a launch of its own (about 2 us).

    Up to M = 8: the form that runs every shape. Up to M = 16: 16 columns and 4 to 16 waves a workgroup
    where that is one round over the CUs (16 waves with their rows of x take a CU's LDS) and K is at most
    4096. Measured on MI355X at M = 12, conversion included, GEMV / tile: 3584 x 3584 7.5 / 8.3 us, 896 x
    896 5.0 / 6.1, 9728 x 896 6.1 / 8.3; two rounds 4608 x 3584 13.1 / 10.3, 9728 x 1536 10.8 / 9.5; long
    K 3584 x 5632 10.2 / 10.1, 3584 x 11008 15.3 / 13.7."""
    if m <= STREAM_WIDE_M:
        return split_k_gemv_config(n, k)
    waves = _pow2_at_most(k // 128, 16)
    if m <= W4A8_GEMV_MAX_M and k <= 4096 and -(-n // 16) * waves <= 16 * NUM_CUS:
        return GemmConfig("gemv_mfma", 16, 16, 128, 1, waves, 2)
    return None


# Makespan model of the fp8 GEMM on MI355X (fit to its measured times on the Qwen2.5-7B shapes):
# a workgroup runs one 128-K block of a BM x BN tile at about 4.2 TFLOP/s, the 256 x 160 tile 5%
# slower per FLOP; a K split adds about 3 us plus its fp32 partials (split * M * N * 4 bytes
# written and read back) at about 4 TB/s.
_FP8_CU_FLOP_PER_US = 4.2e6
_FP8_SPLIT_US = 3.0
_FP8_PARTIAL_BYTES_PER_US = 4.0e6


@functools.lru_cache(maxsize=None)
def fp8_gemm_config(bucket: int, n: int, k: int) -> GemmConfig:
    """Launch config of the W4A8 fp8 GEMM for one bucket: the tile and K split with the lowest
    modelled time (rounds of workgroups over the CUs x blocks per workgroup x block time, plus
    the split's partials), in its producer / consumer form where the tile has one. On the
    Qwen2.5-7B shapes it picks the configs measured fastest: gate_up 256 x 160 at M = 256 and
    256 x 128 above; down 256 x 128 with split 9 / 2 / 1 at M = 256 / 1024 / 4096."""
    tiles_by_m = ((256, 128), (256, 160), (256, 192)) if bucket >= 256 else ((128, 256), (128, 128))
    k_blocks = max(1, k // 128)
    best: tuple[float, int, int, int] | None = None
    for bm, bn in tiles_by_m:
        tiles = -(-n // bn) * -(-bucket // bm)
        block_us = bm * bn * 128 * 2 / _FP8_CU_FLOP_PER_US * (1.05 if bn == 160 else 1.0)
        # Powers of two, and the split that fills the CUs in whole rounds (fill_split; with
        # 28 column tiles of down_proj, split 9 is 3% faster than 8 at M = 128 and 256).
        fill = fill_split(GemmConfig("gemm_fp8", bm, bn, 128, 1, 8, 3), bucket, n, k, NUM_CUS)
        for split in sorted({1, 2, 4, 8, fill}):
            if split > 1 and split * 4 > k_blocks:
                break
            rounds = -(-tiles * split // NUM_CUS)
            us = rounds * -(-k_blocks // split) * block_us
            if split > 1:
                us += _FP8_SPLIT_US + split * bucket * n * 8 / _FP8_PARTIAL_BYTES_PER_US
            if best is None or us < best[0]:
                best = (us, bm, bn, split)
    assert best is not None
    _, bm, bn, split = best
    # the producer / consumer form where the tile has one (same box, Qwen2.5-7B shapes: 3-14%
    # faster than the shared-role form at M = 256..4096)
    stages = 8 if any((bm, bn) == (pbm, pbn) for pbm, pbn, _, _ in FP8_PC_TILES) else 3
    return GemmConfig("gemm_fp8", bm, bn, 128, split, 8, stages)
