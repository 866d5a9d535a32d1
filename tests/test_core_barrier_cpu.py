"""The peeling kernel's grid barrier, as compiled: every wave must have waited for
its own memory operations when its block arrives.  A wave's stores and its adds
that return nothing are in flight across a block barrier, and blocks on other
XCDs read them (degrees, overflow entries) as soon as the grid barrier opens, so
the wait has to stand between the last of them and the block barrier.  A missing
one cannot be shown by running: it shows in the compiled code."""

import os
import re
import shutil
import subprocess

import pytest

from scs_amd import build

KERNEL = "core_peel"


def kernel_lines(text, kernel):
    lines = text.splitlines()
    start = next(i for i, s in enumerate(lines) if re.match(rf"_Z\d+{kernel}\w*:", s))
    end = next(i for i in range(start, len(lines)) if lines[i].startswith(".Lfunc_end"))
    # instructions and labels, without comments and directives
    out = [re.split(r"[;]|//", s)[0].strip() for s in lines[start:end]]
    return [s for s in out if s and not (s.startswith(".") and not s.endswith(":"))]


def waits_before(lines, i):
    """Whether vmcnt(0) stands before line i, after the last vector memory
    operation, label or branch."""
    for s in reversed(lines[:i]):
        if s.startswith("s_waitcnt") and "vmcnt(0)" in s:
            return True
        if s.endswith(":") or re.match(r"(global|flat|buffer|scratch)_|s_(cbranch|branch)", s):
            return False
    return False


def test_every_wave_waits_before_its_block_arrives(tmp_path):
    if not (os.path.exists(build.HIPCC) or shutil.which(build.HIPCC)):
        pytest.skip("no hipcc")
    asm = tmp_path / "graph.s"
    subprocess.run([build.HIPCC, f"--offload-arch={build.ARCH}", "-O3", "-std=c++17",
                    *build.DEV_FLAGS, "--offload-device-only", "-S", "-o", str(asm),
                    os.path.join(build.CSRC, "scs_graph.hip")], check=True, capture_output=True)
    lines = kernel_lines(asm.read_text(), KERNEL)
    barriers = [i for i, s in enumerate(lines) if s.startswith("s_barrier")]
    # a block barrier whose next 64-bit add is an arrival: no barrier between
    arrivals = []
    for b, nxt in zip(barriers, barriers[1:] + [len(lines)]):
        if any(s.startswith("global_atomic_add_x2") for s in lines[b:nxt]):
            arrivals.append(b)
    assert arrivals
    for b in arrivals:
        assert waits_before(lines, b), "no vmcnt(0) before the barrier at " + str(lines[b - 4:b + 1])
