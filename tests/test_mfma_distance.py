"""Distance between an MFMA and the reads of its result, checked on the built code.

The hardware does not hold a vector or memory instruction back that reads an
MFMA's result too early; the compiler fills the distance up (8 wait states after
the 16x16x32 forms, 10 after the f32 16x16x4), but has been seen to leave one or
two where the read lies behind a taken branch (ops.hpp, mfma_pin).  This test
disassembles the library's gfx950 code objects and follows every path from every
MFMA to the first such read.
"""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tang_amd", "libtang_hip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
NEEDED = {"v_mfma_f32_16x16x4_f32": 10}
DEFAULT = 8


def _regs(text):
    out = set()
    for kind, lo, hi, k1, n in re.findall(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", text):
        if kind:
            out.update(kind + str(i) for i in range(int(lo), int(hi) + 1))
        else:
            out.add(k1 + n)
    return out


def _decode(line, labels):
    """(opcode, registers written, registers read, wait states, branch target)"""
    text, _, note = line.partition("//")
    op, _, args = text.strip().partition(" ")
    args = args.strip()
    parts = re.split(r",\s*(?![^\[]*\])", args)
    writes = "store" in op or op.startswith(("ds_write", "global_atomic", "buffer_atomic", "v_cmp"))
    dst = set() if writes else _regs(parts[0])
    src = _regs(args if writes else ",".join(parts[1:]))
    if op.startswith(("v_fmac", "v_mac", "v_pk_fmac", "v_dot2c")):
        src |= dst
    target = None
    if op.startswith(("s_branch", "s_cbranch")):
        m = re.search(r"\+0x([0-9a-f]+)>", note)
        target = labels.get(int(m.group(1), 16) if m else 0)
    return op, dst, src, int(args.split()[0]) + 1 if op == "s_nop" else 1, target


def short_reads(lines):
    """Reads of an MFMA's result that lie too close to it on some path.  lines:
    a kernel's instructions as (offset, text)."""
    labels = {off: i for i, (off, _) in enumerate(lines)}
    code = [_decode(t, labels) for _, t in lines]
    bad = []
    for i, (op, dst, _, _, _) in enumerate(code):
        if "mfma" not in op:
            continue
        need = NEEDED.get(re.sub(r"_e\d\d$", "", op), DEFAULT)
        seen, todo = {}, [(i + 1, 0, frozenset(dst))]
        while todo:
            j, dist, live = todo.pop()
            if j is None or j >= len(code) or dist >= need or not live or seen.get((j, live), need) <= dist:
                continue
            seen[j, live] = dist
            o, d, s, states, target = code[j]
            if live & s and "mfma" not in o:  # an MFMA that reads it waits by itself
                bad.append("%s, %d states later: %s" % (lines[i][1].split("//")[0].strip(), dist,
                                                        lines[j][1].split("//")[0].strip()))
                continue
            if o == "s_endpgm":
                continue
            if target is not None:
                todo.append((target, dist + states, live - d))
            if o != "s_branch":
                todo.append((j + 1, dist + states, live - d))
    return bad


def test_short_reads_follows_branches():
    """One state behind a taken branch is found, the same behind its wait is not."""
    k = [(0, "v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[8:11], 0"),
         (8, "s_cbranch_scc1 1 // 0: <k+0x10>"),
         (12, "s_nop 9"),
         (16, "v_add_f32_e32 v4, v5, v1")]
    assert len(short_reads(k)) == 1
    assert not short_reads(k[:1] + [(8, "s_nop 6"), (12, "s_cbranch_scc1 0 // 0: <k+0x10>")] + k[3:])
    assert len(short_reads(k[:1] + [(8, "ds_write_b32 v20, v2")])) == 1


@pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(LIB)), reason="needs llvm-objdump and the built library")
def test_no_mfma_result_is_read_early(tmp_path):
    lib = str(tmp_path / "lib.so")
    shutil.copy(LIB, lib)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True, cwd=str(tmp_path))
    bad, mfmas = [], 0
    for b in tmp_path.iterdir():
        if not b.name.endswith("gfx950"):
            continue
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(b)], check=True, capture_output=True, text=True).stdout
        for sym in re.split(r"^(?=[0-9a-f]+ <)", out, flags=re.M):
            if "v_mfma" not in sym:
                continue
            head, *body = sym.splitlines()
            lines = []
            for line in body:
                m = re.match(r"\s+(\S.*// ([0-9A-F]+):.*)$", line)
                if m:
                    lines.append((int(m.group(2), 16) - int(head.split()[0], 16), m.group(1)))
            mfmas += sum("v_mfma" in t for _, t in lines)
            bad += ["%s: %s" % (head.split()[1][:100], x) for x in short_reads(lines)]
    assert mfmas > 1000
    assert not bad, "\n".join(bad[:20])
