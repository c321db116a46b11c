"""The K-split tile GEMM's hand-written waits on its generated gfx950 code: every block barrier's
vmcnt(N) is at most the loads issued after the x stage it guards, on every control-flow path (the
walk of ``test_isa_order``). Needs hipcc, no GPU."""

from __future__ import annotations

import re
import subprocess
from pathlib import Path

import pytest

from tests.unit.test_isa_order import CSRC, _instructions, _order_after_barriers, _wait_checks
from tokenforge_amd import build

X_STAGES = 2
_KERNEL = re.compile(r"^(_Z\w*gemm5_kernelI(\w*?)EEv\w*):")


def test_ksplit_stage_waits(tmp_path: Path) -> None:
    try:
        cc = build.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not available")
    out = tmp_path / "gemm5.s"
    flags = [f for f in build.HIPCC_FLAGS if f != "-fPIC"]
    subprocess.run([cc, *flags, "--cuda-device-only", "-S", str(CSRC / "gemm5.hip"), "-o", str(out)], check=True,
                   capture_output=True)
    asm = out.read_text()
    good, bad = _order_after_barriers(asm)
    assert good > 0 and bad == 0
    lines = asm.splitlines()
    kernels = 0
    for i, line in enumerate(lines):
        m = _KERNEL.match(line)
        if not m:
            continue
        end = next(j for j in range(i + 1, len(lines)) if lines[j].startswith(".Lfunc_end"))
        rows = _wait_checks(_instructions(lines[i + 1:end]), X_STAGES)
        assert len(rows) >= 2, m.group(1)
        for b, n, after in rows:
            assert after >= 0 and after != float("inf"), f"{m.group(1)}: barrier at {b}"
            assert n <= after, f"{m.group(1)}: barrier at {b} waits vmcnt({n}), only {after} loads follow the stage"
        kernels += 1
    assert kernels > 0
