"""Waits in kernel sources are pinned: the wait builtin does not tell the
compiler that it orders memory, so an access may be moved past it."""

import re
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "vllm_amd" / "csrc"
BARRIER = 'asm volatile("" ::: "memory");'


def test_waits_lie_between_compiler_barriers():
    """The builtin is called in common.h only; there with a barrier on both
    sides, except for fills (volatile statements themselves, which stay in
    order with it)."""
    for path in sorted(CSRC.glob("*.h")) + sorted(CSRC.glob("*.hip")):
        lines = [l.split("//")[0].strip() for l in
                 path.read_text().splitlines()]
        for i, line in enumerate(lines):
            if "__builtin_amdgcn_s_waitcnt" not in line:
                continue
            where = f"{path.name}:{i + 1}"
            assert path.name == "common.h", where
            if re.search(r"N & 15", line):   # lds_fill_wait
                continue
            assert lines[i - 1] == BARRIER, where
            after = i + 1 + ("s_barrier" in lines[i + 1])
            assert lines[after] == BARRIER, where
