"""What the block form's kernels (fdtd2d_amd/csrc/block_device.h) take from the
compiler without the language promising it, checked in the assembly of this
repository's own build (hipcc cross-compiles, no GPU needed):

* every barrier is behind a wait for the wave's LDS writes, with no LDS write
  between them: a neighbour reads those rows right after the barrier;
* no readlane takes a register that was last reloaded from a spill: a reload
  under a partial mask leaves the other lanes as they were, and an address or a
  row number read from one of those lanes is garbage."""

from __future__ import annotations

import re
import subprocess
from pathlib import Path

import pytest

from fdtd2d_amd import build

HIPCC = Path(build.HIPCC)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """The instructions of each block kernel, in order."""
    if not HIPCC.exists():
        pytest.skip("needs hipcc")
    out = tmp_path_factory.mktemp("asm") / "block.s"
    subprocess.run([str(HIPCC), *build.HIPFLAGS, "--cuda-device-only", "-S",
                    str(build.CSRC / "block_kernels.hip"), "-o", str(out)], check=True, capture_output=True, text=True,
                   timeout=300)
    found, name = {}, None
    for line in out.read_text().splitlines():
        start = re.match(r"(_Z\w*block\w*kernel\w*):", line)
        if start:
            name = start.group(1)
            found[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name:
            ins = line.split(";")[0].strip()
            if ins and not ins.startswith(".") and not ins.endswith(":"):
                found[name].append(ins)
    return found


def unguarded_barriers(code):
    """Barriers with no wait for LDS between them and the last LDS write."""
    bad = 0
    for i, ins in enumerate(code):
        if not ins.startswith("s_barrier"):
            continue
        for prev in reversed(code[:i]):
            if prev.startswith("s_waitcnt") and "lgkmcnt(0)" in prev:
                break
            if prev.startswith(("ds_write", "ds_store", "s_barrier", "s_cbranch", "s_branch")):
                bad += 1
                break
    return bad


def reloads_read_across_lanes(code):
    """readlane and readfirstlane instructions whose source was last written by
    a reload: from scratch, or from an accumulation register."""
    reloaded, bad = set(), []
    for ins in code:
        op, _, rest = ins.partition(" ")
        args = [a.strip() for a in rest.split(",")]
        if op.startswith(("v_readlane", "v_readfirstlane")):
            if args[1] in reloaded:
                bad.append(ins)
            continue
        dst = re.fullmatch(r"v(\d+)|v\[(\d+):(\d+)\]", args[0]) if args else None
        if not dst or op.startswith(("scratch_store", "global_store", "buffer_store", "ds_write", "v_cmp")):
            continue
        lo, hi = (int(dst.group(1)),) * 2 if dst.group(1) else (int(dst.group(2)), int(dst.group(3)))
        regs = {f"v{r}" for r in range(lo, hi + 1)}
        reloaded = reloaded | regs if op.startswith(("scratch_load", "v_accvgpr_read")) else reloaded - regs
    return bad


def test_checks_see_planted_mistakes():
    good = ["ds_write_b32 v1, v2", "s_waitcnt lgkmcnt(0)", "s_barrier"]
    assert unguarded_barriers(good) == 0
    assert unguarded_barriers([good[0], good[2]]) == 1
    assert unguarded_barriers([good[1], good[0], good[2]]) == 1
    assert unguarded_barriers(["s_waitcnt vmcnt(0)", "s_cbranch_scc1 .LBB0_1", "s_barrier"]) == 1
    assert reloads_read_across_lanes(["scratch_load_dword v7, off, off offset:4", "v_readlane_b32 s3, v7, 1"])
    assert reloads_read_across_lanes(["scratch_load_dwordx2 v[6:7], off, off", "v_readfirstlane_b32 s3, v7"])
    assert not reloads_read_across_lanes(["scratch_load_dword v7, off, off", "v_mov_b32_e32 v7, v8",
                                          "v_readlane_b32 s3, v7, 1"])


def test_barriers_wait_for_the_lds_writes(kernels):
    # plans and pools, {2,4,4,12} for the density medium, two shapes for both
    assert len(kernels) == 10
    for name, code in kernels.items():
        assert sum(i.startswith("s_barrier") for i in code) >= 5, name
        assert unguarded_barriers(code) == 0, name


def test_no_readlane_of_a_reloaded_register(kernels):
    assert sum(i.startswith("v_readlane") for code in kernels.values() for i in code) > 100
    for name, code in kernels.items():
        assert not reloads_read_across_lanes(code), name
