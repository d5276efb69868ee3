"""What the kernels' sources promise and no run shows reliably."""
import glob
import os
import re

import pytest

from litellmengine_amd.csrc import build

SOURCES = sorted(glob.glob(os.path.join(os.path.dirname(build.__file__), "*.hip")))


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_bare_barriers_wait_for_lds(path):
    """A bare s_barrier waits for nothing: without lgkmcnt(0) ahead of it a wavefront's reads from LDS may still be on their way
    when another one, behind the barrier, fills the buffer anew.  Every path to it has that wait (or a release fence on LDS)."""
    lines = [re.sub(r"//.*", "", line).strip() for line in open(path)]
    lines = [line for line in lines if line]
    for i, line in enumerate(lines):
        if "__builtin_amdgcn_s_barrier()" not in line or line.startswith("#"):
            continue
        before, at = [], i - 1
        while at >= 0 and re.match(r"(if|else|asm volatile\(\"s_waitcnt|__builtin_amdgcn_fence\(__ATOMIC_RELEASE)", lines[at]):
            before.append(lines[at])
            at -= 1
        waits = [w for w in before if "s_waitcnt" in w or "fence" in w]
        assert waits, f"{os.path.basename(path)}: {lines[at]} / {line}"
        assert all("lgkmcnt(0)" in w or "fence" in w for w in waits), (os.path.basename(path), waits)
