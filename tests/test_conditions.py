"""The built kernels, as the disassembler lists them: no scalar instruction
takes a condition (SCC) that its own block has not set.

A 64-bit comparison that only the vector ALU has may become a select of the
scalar ALU without the copy of its result between them. What the select then
takes is the condition of whatever was compared last, in another block."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

from test_product_waits import _code_objects

READS = re.compile(r"s_(cselect_b|cbranch_scc|addc_u32|subb_u32|cmov)")
SETS = re.compile(
    r"s_(add|sub|addc|subb|addk|abs|absdiff|min|max|and|or|xor|not|andn1|andn2"
    r"|orn1|orn2|nand|nor|xnor|lshl|lshr|ashr|bfe|bcnt0|bcnt1|cmp|cmpk|bitcmp"
    r"|quadmask|wqm|lshl[1-4]_add)(_|\d)|s_\w+_saveexec|s_andn[12]_wrexec")


def strays(lines):
    """Of one kernel: [(instruction, the one before it)]."""
    ops, at, jumps = [], {}, []
    for line in lines:
        m = re.match(r"\s+(\S+)(.*?)//\s*([0-9A-Fa-f]+):(.*)", line)
        if not m:
            continue
        name, rest, addr, tail = m.groups()
        at[int(addr, 16)] = len(ops)
        t = re.search(r"<[^>]*\+0x([0-9a-fA-F]+)>", tail)
        if "branch" in name:
            jumps.append(int(t.group(1), 16) if t else 0)
        ops.append((name, (name + rest).strip()))
    if not ops:
        return []
    base = min(at)
    joins = {at[base + off] for off in jumps}
    found, known = [], False
    for i, (name, text) in enumerate(ops):
        # What falls through a branch keeps the condition.
        if i in joins or (i and ops[i - 1][0].startswith(
                ("s_branch", "s_endpgm", "s_setpc", "s_swappc"))):
            known = False
        if READS.match(name) and not known:
            found.append((text, ops[i - 1][1] if i else ""))
        if SETS.match(name):
            known = True
    return found


def test_built_kernels_take_their_own_conditions(tmp_path):
    import vllm_amd
    library = Path(vllm_amd.__file__).parent / "_C.so"
    objdump = shutil.which("llvm-objdump",
                           path="/opt/rocm/llvm/bin:/opt/rocm/bin")
    if not library.exists() or objdump is None:
        pytest.skip("extension or disassembler not there")
    kernels = 0
    for i, code in enumerate(_code_objects(library)):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", path],
                              check=True, capture_output=True,
                              text=True).stdout
        name, lines = None, []
        for line in text.splitlines() + ["0 <>:"]:
            m = re.match(r"[0-9a-f]+ <(\S*)>:", line)
            if not m:
                lines.append(line)
                continue
            if name is not None:
                kernels += 1
                assert strays(lines) == [], name
            name, lines = m.group(1), []
    assert kernels > 100


def _listed(*ops):
    """Four bytes each; a branch goes to the operation of its number."""
    return [f"\t{op.split(' -> ')[0]} // {i * 4:012X}: "
            + (f"<k+0x{int(op.split(' -> ')[1]) * 4:x}>" if "->" in op else "")
            for i, op in enumerate(ops)]


@pytest.mark.parametrize("ops,n", [
    (["s_cmp_lg_u32 s0, 0", "s_cselect_b32 s0, s1, 32"], 0),
    (["s_cmp_lg_u32 s0, 0", "s_mov_b32 s2, 0", "s_addc_u32 s0, s1, s2"], 0),
    (["s_ff1_i32_b32 s0, s1", "s_cselect_b32 s0, s0, 32"], 1),
    # Behind a branch, and where another path joins.
    (["s_cmp_lg_u32 s0, 0", "s_cbranch_scc0 2 -> 3", "s_cselect_b32 s0, s1, 2",
      "s_endpgm"], 0),
    (["s_cmp_lg_u32 s0, 0", "s_cbranch_scc0 2 -> 3", "s_cmp_eq_u32 s1, 0",
      "v_cmp_gt_u64_e32 vcc, s[0:1], v[2:3]", "s_cselect_b32 s0, s1, 2"], 1),
    (["s_cmp_lg_u32 s0, 0", "s_branch 1 -> 3", "s_cmov_b32 s0, s1",
      "s_endpgm"], 1)])
def test_strays(ops, n):
    assert len(strays(_listed(*ops))) == n
