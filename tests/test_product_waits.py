"""Matrix products written as inline assembly (csrc/common.h: mfma16_acc) are
outside what the compiler pads with waits: a register that it moves right
before or after one would be read too early, with no error. These tests read
the instructions of the built kernels and look at every path through them."""

import re
import shutil
import struct
import subprocess
from collections import deque
from pathlib import Path

import pytest

# Wait states that must lie between an instruction that is no matrix product
# and writes a register, and a product that reads it; and between a product
# and any other instruction that touches what it writes, or a product that
# reads it as an operand. The least that the compiler leaves around the
# products it knows, in all kernels of this library.
BEFORE = 2
AFTER = {"16x16x32": 8, "32x32x16": 12}
CAP = max(AFTER.values())

KERNELS = ("tile_linear_kernel", "moe_tile_kernel")

_REG = re.compile(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])")


def _regs(text):
    out = []
    for kind, one, lo, hi in _REG.findall(text):
        a, b = (int(one), int(one)) if one else (int(lo), int(hi))
        out.append(frozenset((kind, i) for i in range(a, b + 1)))
    return out


def _after(name):
    for shape, states in AFTER.items():
        if shape in name:
            return states
    return CAP


class _Op:
    """One instruction: what it does to the two tables of ages."""

    def __init__(self, name, rest):
        self.text = f"{name} {rest}"
        self.name = name
        self.states = int(rest.split()[0], 0) + 1 if name == "s_nop" else 1
        self.product = name.startswith("v_mfma")
        regs = _regs(rest)
        self.touches = frozenset().union(*regs)
        self.writes = frozenset()
        if self.product:
            self.writes = regs[0]
            # A sum may go on at once.
            self.touches = frozenset().union(*regs[1:3])
        elif name.startswith("v_") and regs:
            first = rest.split(",")[0]
            if "swap" in name:
                self.writes = regs[0] | regs[1]
            elif _REG.search(first):
                self.writes = regs[0]
        self.reads_c = regs[3] if self.product and len(regs) > 3 \
            else frozenset()


def _step(op, valu, mfma, say):
    """Ages after `op`, from those before it."""
    if op.product:
        for r in op.touches | op.reads_c:
            if valu.get(r, BEFORE) < BEFORE:
                say(op, f"{r} written {valu[r]} states before")
    for r in op.touches:
        if r in mfma and mfma[r][0] < mfma[r][1]:
            say(op, f"{r}: {mfma[r][0]} states after a product")
    n = op.states
    valu = {r: a + n for r, a in valu.items() if a + n < BEFORE}
    mfma = {r: (a + n, w) for r, (a, w) in mfma.items() if a + n < w}
    if op.product:
        for r in op.writes:
            mfma[r] = (0, _after(op.name))
            valu.pop(r, None)
    else:
        for r in op.writes:
            valu[r] = 0
            mfma.pop(r, None)
    return valu, mfma


def _join(old, new):
    """The younger age of every register; whether that is news."""
    if old is None:
        return new, True
    valu, mfma = dict(old[0]), dict(old[1])
    news = False
    for r, a in new[0].items():
        if a < valu.get(r, BEFORE):
            valu[r], news = a, True
    for r, (a, w) in new[1].items():
        have = mfma.get(r)
        if have is None or have[1] - have[0] < w - a:
            mfma[r], news = (a, w), True
    return (valu, mfma), news


def violations(lines):
    """Of one kernel as llvm-objdump lists it: [(instruction, why)]."""
    ops, at, jump = [], {}, {}
    for line in lines:
        m = re.match(r"\s+(\S+)(.*?)//\s*([0-9A-Fa-f]+):(.*)", line)
        if not m:
            continue
        name, rest, addr, tail = m.groups()
        at[int(addr, 16)] = len(ops)
        t = re.search(r"<[^>]*\+0x([0-9a-fA-F]+)>", tail)
        if "branch" in name:
            jump[len(ops)] = int(t.group(1), 16) if t else 0
        ops.append(_Op(name, rest.strip()))
    if not ops:
        return []
    base = min(at)
    target = {i: at[base + off] for i, off in jump.items()}
    starts = sorted({0, *target.values(), *(i + 1 for i in jump)})
    starts = [s for s in starts if s < len(ops)]
    end_of = dict(zip(starts, starts[1:] + [len(ops)]))
    state = {0: ({}, {})}
    todo, found = deque([0]), {}
    while todo:
        b = todo.popleft()
        cur = state[b]
        for i in range(b, end_of[b]):
            cur = _step(ops[i], *cur,
                        lambda op, why: found.setdefault((i, why), op.text))
        last = end_of[b] - 1
        nexts = []
        if last in target:
            nexts.append(target[last])
        if not ops[last].name.startswith(("s_branch", "s_endpgm", "s_setpc")) \
                and last + 1 < len(ops):
            nexts.append(last + 1)
        for n in nexts:
            state[n], news = _join(state.get(n), cur)
            if news:
                todo.append(n)
    return [(text, why) for (_, why), text in sorted(found.items())]


def _code_objects(library):
    """The gfx950 code objects in a shared library."""
    data = library.read_bytes()
    mark = b"__CLANG_OFFLOAD_BUNDLE__"
    at = data.find(mark)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length]
            p += 24 + length
            if size and name.endswith(b"gfx950"):
                yield data[at + off:at + off + size]
        at = data.find(mark, at + 24)


def _listing(tmp_path):
    """{kernel: its lines} of the kernels named above."""
    import vllm_amd
    library = Path(vllm_amd.__file__).parent / "_C.so"
    objdump = shutil.which("llvm-objdump",
                           path="/opt/rocm/llvm/bin:/opt/rocm/bin")
    if not library.exists() or objdump is None:
        pytest.skip("extension or disassembler not there")
    out = {}
    for i, code in enumerate(_code_objects(library)):
        if not any(k.encode() in code for k in KERNELS):
            continue
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        text = subprocess.run([objdump, "-d", "--no-show-raw-insn", path],
                              check=True, capture_output=True,
                              text=True).stdout
        cur = None
        for line in text.splitlines():
            m = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if m:
                cur = out.setdefault(m.group(1), []) \
                    if any(k in m.group(1) for k in KERNELS) else None
            elif cur is not None:
                cur.append(line)
    return out


def test_built_kernels_wait(tmp_path):
    kernels = _listing(tmp_path)
    for k in KERNELS:
        assert any(k in name for name in kernels)
    for name, lines in kernels.items():
        assert any("v_mfma" in line for line in lines), name
        assert violations(lines) == [], name


def _lines(*ops):
    """A listing of these instructions; "-> n" after one jumps to the n-th."""
    out = []
    for i, op in enumerate(ops):
        op, _, to = op.partition(" -> ")
        where = f" <kernel+0x{8 * int(to):x}>" if to else ""
        out.append(f"\t{op}  // {4096 + 8 * i:012X}: 00000000{where}")
    return out


PRODUCT = "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]"


@pytest.mark.parametrize("ops,clean", [
    # A chain in place, and what it may be read and moved behind.
    ([PRODUCT, PRODUCT, "s_nop 7", "v_accvgpr_read_b32 v9, a1"], True),
    ([PRODUCT, "s_nop 6", "v_accvgpr_read_b32 v9, a1"], False),
    ([PRODUCT, "v_accvgpr_read_b32 v9, a4"], True),
    ([PRODUCT, "v_accvgpr_mov_b32 a3, a9"], False),
    ([PRODUCT, "global_store_dwordx4 v[10:11], a[0:3], off"], False),
    # An accumulator or an operand that a move writes right before.
    (["v_accvgpr_write_b32 a2, 0", "s_nop 1", PRODUCT], True),
    (["v_accvgpr_write_b32 a2, 0", "s_nop 0", PRODUCT], False),
    (["v_mov_b32_e32 v5, v20", PRODUCT], False),
    (["v_mov_b32_e32 v5, v20", "s_nop 1", PRODUCT], True),
    (["v_permlane16_swap_b32_e32 v20, v5", PRODUCT], False),
    (["v_cmp_gt_u32_e32 vcc, v5, v20", PRODUCT], True),
    # A product as another's operand.
    (["v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[12:15], 0", PRODUCT],
     False),
    # Round a loop: the move at its end meets the product at its start.
    (["s_nop 1", PRODUCT, "s_nop 7", "v_accvgpr_write_b32 a2, 0",
      "s_cbranch_scc0 65533 -> 1", "s_endpgm"], False),
    (["s_nop 1", PRODUCT, "s_nop 7", "v_accvgpr_write_b32 a2, 0",
      "s_cbranch_scc0 65533 -> 0", "s_endpgm"], True),
    # By one of two ways only.
    (["s_cbranch_scc0 2 -> 3", PRODUCT, "s_branch 1 -> 4", "s_nop 7",
      "v_accvgpr_read_b32 v9, a1", "s_endpgm"], False),
    (["s_cbranch_scc0 2 -> 3", PRODUCT, "s_endpgm", "s_nop 0",
      "v_accvgpr_read_b32 v9, a1", "s_endpgm"], True),
])
def test_violations(ops, clean):
    assert (violations(_lines(*ops)) == []) == clean
